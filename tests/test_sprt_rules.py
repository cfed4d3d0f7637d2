"""The SPRT walk on the host: tests/cpp/sprt_check.cpp compiled against the
headers that the kernels are built from (csrc/sprt_rules.hpp, csrc/dev_sprt.hpp)."""
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
    subprocess.check_call([gxx, "-std=c++17", "-O2", "-ffp-contract=off", "-Wno-unknown-pragmas", "-o", exe,
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


@pytest.mark.parametrize("order", ["pool", "cells"])
def test_walk_matches_the_products_one_by_one(check, order):
    """The kernel's walk of a model, its 64 lanes run as contexts, against the
    reference's loop over positions: count, tested points, decision and, over
    cells, the tested inliers.  Random bits, cells and parameters; thresholds
    exactly at a product, below 1, infinite, NaN and negative; equal and nearly
    equal delta and epsilon; runs that sink the product below the normal range
    and bring it back; rows beyond the 64 words that the lanes hold."""
    check(order)
