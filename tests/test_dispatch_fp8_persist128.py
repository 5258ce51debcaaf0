"""The dispatch rule between the fp8 dot's 128 x 128 persistent tile and its
256 x 128 tile with K split (fp8_persist128 in tx_op_dot.cpp), on the CPU: the
rule is taken from the source and compiled by itself, for 256 CUs.

MEASURED holds products timed on both tiles on one MI355X, plain, with bias and
with bias + silu (microseconds: 256 x 128 tile, 128 x 128 tile): the rule may
not pick a side that is more than 2% slower.  The shapes that the GPU tests of
the tile name have to reach it.
"""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-ext_amd", "csrc", "host",
                   "tx_op_dot.cpp")
MEASURED = {
    # M, N, K:              plain           bias            bias + silu
    (1536, 6144, 1024): ((21.3, 19.2), (26.1, 30.0), (31.5, 37.7)),
    (1700, 5000, 1024): ((20.1, 17.5), (25.7, 28.5), (31.7, 37.5)),
    (2000, 6000, 768): ((18.6, 16.4), (24.1, 27.1), (30.2, 36.4)),
    (1500, 6000, 512): ((16.5, 14.1), (22.0, 24.7), (28.1, 33.8)),
    (3000, 3000, 3072): ((40.0, 34.8), (45.4, 45.7), (51.8, 55.1)),
    (900, 9000, 4096): ((47.6, 43.7), (53.1, 54.0), (59.6, 63.4)),
    (2304, 5120, 4096): ((52.3, 49.3), (56.1, 56.1), (62.3, 65.9)),
    (3000, 3000, 8192): ((90.9, 81.5), (96.5, 95.6), (102.9, 105.1)),
    (900, 9000, 14336): ((147.8, 137.0), (153.6, 148.7), (160.1, 157.0)),
    (600, 12000, 1024): ((19.5, 13.3), (25.3, 20.8), (31.4, 26.7)),
    (1100, 7168, 2048): ((28.2, 20.4), (34.0, 26.8), (40.1, 32.9)),
    (130, 14336, 1024): ((18.2, 7.9), (24.0, 11.6), (24.9, 14.8)),
    (700, 2048, 2048): ((22.7, 10.2), (25.4, 14.1), (25.9, 17.1)),
    (1024, 4096, 4096): ((30.4, 19.7), (41.0, 21.9), (41.8, 24.8)),
    (256, 4096, 4096): ((22.2, 15.8), (26.8, 19.7), (27.2, 23.3)),
    (2048, 2048, 512): ((9.9, 7.5), (11.9, 10.9), (15.1, 13.9)),
    (65, 14336, 1024): ((13.5, 7.6), (18.2, 11.3), (18.7, 14.4)),
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    with open(SRC) as f:
        text = f.read()
    parts = re.findall(r"^constexpr int64_t (?:kMinStepsPerSplit|kMaxSplits|kEpiRoundSteps) = \d+;", text, re.M)
    parts.append(re.search(r"^bool fp8_persist128\(.*?^}", text, re.M | re.S)[0])
    d = tmp_path_factory.mktemp("rule")
    cpp, so = str(d / "rule.cpp"), str(d / "rule.so")
    with open(cpp, "w") as f:
        f.write("#include <algorithm>\n#include <cstdint>\n" + "\n".join(parts) +
                '\nextern "C" int rule(int64_t M, int64_t N, int64_t steps, bool epi) '
                "{ return fp8_persist128(M, N, steps, 256, epi); }\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", cpp, "-o", so], check=True)
    fn = ctypes.CDLL(so).rule
    fn.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_bool]
    return lambda M, N, K, epi: bool(fn(M, N, K // 128, epi))


@pytest.mark.parametrize("shape", list(MEASURED))
@pytest.mark.parametrize("form", [0, 1, 2])
def test_picks_no_slower_tile(rule, shape, form):
    other, here = MEASURED[shape][form]
    got = (other, here)[rule(*shape, form > 0)]
    assert got <= 1.02 * min(other, here), (shape, form, got)


def test_gpu_tests_reach_the_tile(rule):
    for epi in (False, True):
        for shape in [(65, 128, 256), (129, 1000, 384), (700, 2040, 768), (512, 512, 256), (600, 12000, 256),
                      (600, 12000, 512), (1024, 1024, 512), (512, 2048, 4096)]:
            assert rule(*shape, epi), (shape, epi)
        for shape in [(2049, 2056, 512), (1023, 4104, 1152)]:
            assert not rule(*shape, epi), (shape, epi)
    assert rule(2047, 2048, 512, False) and rule(1500, 6000, 512, False)
    assert -(-600 // 128) * -(-12000 // 128) > 256 and -(-1500 // 128) * -(-6000 // 128) > 512
