"""The SPRT walk's rules (csrc/sprt_rules.hpp, the header the kernels use) on
the host: tests/cpp/sprt_check.cpp compiled against it."""
import os
import shutil
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module")
def check(tmp_path_factory):
    gxx = shutil.which("g++")
    if not gxx:
        pytest.skip("g++ not available")
    exe = str(tmp_path_factory.mktemp("sprt") / "sprt_check")
    subprocess.check_call([gxx, "-std=c++17", "-O2", "-ffp-contract=off", "-o", exe,
                           "-I", os.path.join(ROOT, "graph-cut-ransac_amd", "csrc"),
                           os.path.join(ROOT, "tests", "cpp", "sprt_check.cpp")])

    def run(what):
        r = subprocess.run([exe, what], capture_output=True, text=True, timeout=300)
        assert r.returncode == 0, r.stdout
        print(r.stdout)
    return run


def test_every_window_is_a_valid_launch(check):
    """A window's mask launch has a workgroup per item and model: pairs of a
    word of points and tens of thousands of models each must not ask for 2^32
    threads."""
    check("plan")
