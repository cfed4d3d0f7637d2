"""LDS values that pass between the lanes of one wave without a workgroup
barrier go through wave_lds_handover() (csrc/dev_common.hpp): a wave barrier
alone orders no memory, and a queue without either is right only as long as
the compiler cannot tell two indices apart."""
import glob
import os
import re

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "graph-cut-ransac_amd", "csrc")


def _source(name):
    with open(os.path.join(CSRC, name)) as f:
        return re.sub(r"//[^\n]*", "", f.read())


def test_wave_barriers_come_with_fences():
    bare = {os.path.basename(p): _source(os.path.basename(p)).count("__builtin_amdgcn_wave_barrier")
            for p in glob.glob(os.path.join(CSRC, "*.h*"))}
    assert {k: v for k, v in bare.items() if v} == {"dev_common.hpp": 1}
    body = re.search(r"void wave_lds_handover\(\) \{(.*?)\n\}", _source("dev_common.hpp"), re.S).group(1)
    assert re.findall(r"__ATOMIC_\w+|wave_barrier", body) == ["__ATOMIC_RELEASE", "wave_barrier", "__ATOMIC_ACQUIRE"]


def test_per_wave_queues_are_handed_over():
    # a handover before every read of a queue and one before its places are
    # written again
    for name, least in {"k_score.hip": 6, "k_score_mx.hip": 2}.items():
        assert _source(name).count("wave_lds_handover();") >= least, name
    assert "wave_lds_handover();" in _source("k_fund.hip")
