"""The dispatch rules of the 16-bit dots and of small groups, on the CPU: each
rule is taken from tx_op_dot.cpp and compiled by itself, for 256 CUs, and held
to products timed on both sides on one MI355X (microseconds).  It may not pick
a side that is more than 2% slower.
"""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-ext_amd", "csrc", "host",
                   "tx_op_dot.cpp")


@pytest.fixture(scope="module")
def rules(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    with open(SRC) as f:
        text = f.read()
    parts = re.findall(r"^constexpr int64_t (?:kMinStepsPerSplit|kMaxSplits|kSmallMaxSteps) = \d+;", text, re.M)
    parts += re.findall(r"^constexpr int64_t kPadMinWork16 = .*;", text, re.M)
    parts += re.findall(r"^constexpr int64_t kOrderMaxGroups = \d+;", text, re.M)
    parts += [re.search(rf"^(?:bool|int) {fn}\(.*?^}}", text, re.M | re.S)[0]
              for fn in ("persist_beats_split", "small_persist_tile", "pad16_pays", "grouped_persist128", "grouped_dealt")]
    d = tmp_path_factory.mktemp("rules")
    cpp, so = str(d / "rules.cpp"), str(d / "rules.so")
    with open(cpp, "w") as f:
        f.write("#include <algorithm>\n#include <cstdint>\n" + "\n".join(parts) + """
extern "C" int edge(int64_t M, int64_t N, int64_t K) { return small_persist_tile(M, N, 2 * K, 256); }
extern "C" int pad(int64_t M, int64_t N, int64_t K) { return pad16_pays(M, N, K); }
extern "C" int dealt(int64_t G, int64_t N, int64_t K) { return grouped_dealt(G, N, K); }
extern "C" int small_groups(int64_t G, int64_t M, int64_t N, int64_t K) {
  return grouped_persist128(G, M, N, K, 256);
}
extern "C" int here(int64_t M, int64_t N, int64_t K, bool acc, bool kn) {
  return persist_beats_split(M, N, (2 * K + 127) / 128, edge(M, N, K), 256, acc, kn);
}
""")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", cpp, "-o", so], check=True)
    lib = ctypes.CDLL(so)
    lib.edge.argtypes = [ctypes.c_int64] * 3
    lib.pad.argtypes = [ctypes.c_int64] * 3
    lib.dealt.argtypes = [ctypes.c_int64] * 3
    lib.small_groups.argtypes = [ctypes.c_int64] * 4
    lib.here.argtypes = [ctypes.c_int64] * 3 + [ctypes.c_bool] * 2
    return lib


# M, N, K: the tile's edge, 256 x 128 tile with its split, persistent tile
RAGGED = {
    (1000, 1001, 2112): (64, 40.7, 12.6), (1000, 1001, 8192): (64, 50.0, 33.0), (1020, 1020, 4100): (64, 29.1, 22.7),
    (1020, 1020, 6144): (64, 29.1, 26.2), (1020, 1020, 12288): (64, 38.4, 47.2), (1020, 1020, 16384): (64, 44.3, 61.6),
    (1020, 1022, 12288): (64, 57.2, 47.2), (1000, 2001, 4100): (64, 57.5, 40.8), (1000, 2001, 6144): (64, 58.6, 48.8),
    (1000, 2001, 12288): (64, 77.8, 91.0), (1020, 2044, 2112): (64, 27.6, 20.4), (1020, 2044, 4100): (64, 37.6, 40.9),
    (1020, 2044, 8192): (64, 45.2, 63.2), (1500, 1100, 2112): (64, 24.9, 20.0), (1500, 1100, 4100): (64, 34.2, 41.1),
    (1500, 1100, 16384): (64, 61.7, 120.3), (600, 3004, 2112): (64, 24.5, 20.2), (600, 3004, 6144): (64, 37.4, 48.3),
    (3000, 1004, 2112): (64, 30.9, 28.6), (3000, 1004, 4100): (64, 49.1, 59.7), (1025, 2047, 2112): (64, 43.2, 28.5),
    (1025, 2047, 4100): (64, 55.5, 58.2), (2100, 1900, 2112): (64, 31.2, 36.8), (2100, 1900, 8192): (64, 82.9, 122.3),
    (2000, 2001, 2112): (128, 57.3, 21.6), (2000, 2001, 16384): (128, 147.9, 121.8),
    (2040, 2044, 4100): (128, 57.6, 44.5), (2040, 2044, 16384): (128, 129.1, 123.7),
    (1000, 801, 190): (64, None, None), (2500, 3001, 258): (128, None, None), (1000, 2001, 258): (64, None, None),
}


@pytest.mark.parametrize("shape", list(RAGGED))
def test_ragged_picks_no_slower_tile(rules, shape):
    edge, there, here = RAGGED[shape]
    assert rules.edge(*shape) == edge
    pick = rules.here(*shape, False, False)
    if here is None:  # shapes of the persistent tile's GPU tests have to reach it
        assert pick
    else:
        assert (there, here)[pick] <= 1.02 * min(there, here), (shape, pick)


# tt.dot with its accumulator.  M, N, K, row-major B: edge, split, persistent
ACC = {
    (1000, 1000, 1024, 0): (64, 21.3, 9.3), (1000, 1000, 6144, 0): (64, 29.4, 26.1), (1000, 1000, 16384, 0): (64, 44.8, 57.7),
    (1000, 1000, 8192, 1): (64, 40.5, 35.5), (1000, 1000, 16384, 1): (64, 59.6, 64.9), (1024, 1024, 4096, 0): (64, 27.0, 19.9),
    (1024, 1024, 16384, 0): (64, 46.1, 58.0), (640, 2000, 2048, 0): (64, 25.4, 20.6), (640, 2000, 4096, 0): (64, 29.6, 33.0),
    (640, 2000, 4096, 1): (64, 37.4, 35.3), (640, 2000, 16384, 0): (64, 57.2, 109.0), (640, 2000, 16384, 1): (64, 85.0, 118.5),
    (1020, 2044, 4096, 0): (64, 36.9, 34.0), (1020, 2044, 8192, 0): (64, 49.3, 59.0), (1500, 1100, 2048, 0): (64, 27.7, 20.5),
    (1500, 1100, 8192, 0): (64, 43.5, 58.3), (2048, 2048, 2048, 0): (128, 45.6, 24.2), (2048, 2048, 16384, 0): (128, 137.0, 120.5),
    (2048, 2048, 16384, 1): (128, 158.0, 125.3), (2052, 2048, 2048, 0): (128, 46.0, 37.1), (2052, 2048, 4096, 0): (128, 63.7, 60.7),
    (2052, 2048, 8192, 0): (128, 97.8, 107.4), (2052, 2048, 8192, 1): (128, 109.6, 113.2), (2052, 2048, 16384, 0): (128, 171.0, 205.1),
    (2304, 2304, 4096, 0): (128, 69.7, 61.8), (2304, 2304, 8192, 0): (128, 107.5, 109.6), (2304, 2304, 16384, 0): (128, 187.7, 209.1),
    (2304, 2304, 16384, 1): (128, 255.3, 219.4), (3000, 1000, 2048, 0): (64, 34.1, 27.9), (3000, 1000, 4096, 0): (64, 44.6, 46.8),
    (3000, 1000, 4096, 1): (64, 49.6, 51.9), (3000, 1000, 16384, 1): (64, 122.5, 183.8), (1024, 1028, 2048, 0): (64, 26.4, 21.6),
    (1024, 1028, 4096, 0): (64, 30.3, 34.4), (1024, 1028, 16384, 0): (64, 51.0, 109.5), (2048, 3072, 8192, 0): (128, 118.3, 110.7),
    (600, 4000, 4096, 0): (64, 41.6, 46.6), (600, 4000, 4096, 1): (64, 54.9, 47.2), (600, 4000, 16384, 0): (64, 99.7, 160.5),
    # shapes of the persistent tile's GPU tests
    (100, 260, 64 * 21, 0): (64, None, None), (65, 264, 64 * 8, 1): (64, None, None), (129, 4100, 64 * 9, 0): (64, None, None),
    (63, 8, 128, 1): (64, None, None), (1200, 2000, 64 * 9, 0): (64, None, None), (1200, 2000, 64 * 9, 1): (64, None, None),
    (2047, 2044, 64 * 9, 0): (128, None, None), (2048, 2040, 64 * 9, 1): (128, None, None), (2001, 2052, 128, 0): (128, None, None),
}


@pytest.mark.parametrize("case", list(ACC))
def test_accumulating_picks_no_slower_tile(rules, case):
    M, N, K, kn = case
    edge, there, here = ACC[case]
    assert rules.edge(M, N, K) == edge
    pick = rules.here(M, N, K, True, bool(kn))
    if here is None:
        assert pick
    else:
        assert (there, here)[pick] <= 1.02 * min(there, here), (case, pick)


def test_accumulating_form_asks_the_rule():
    with open(SRC) as f:
        body = re.search(r"^static tx_status launch_acc_persist\(.*?^}", f.read(), re.M | re.S)[0]
    assert "!any_k && !persist_beats_split(M, N, (kb + 127) / 128, bt, cus, true, kn)" in body


# odd K below 1 Gi multiply-adds.  M, N, K: generic tile, copies and fast tile
ODD_K = {
    (1000, 1000, 97): (12.0, 14.1), (1000, 1000, 161): (17.3, 13.8), (1500, 1500, 33): (9.5, 18.0),
    (1500, 1500, 97): (12.4, 14.7), (1500, 1500, 161): (17.8, 15.5), (2000, 2000, 17): (9.4, 14.0),
    (2000, 2000, 97): (13.1, 14.2), (2000, 2000, 193): (20.6, 14.6), (2100, 2100, 33): (10.8, 21.5),
    (2100, 2100, 97): (17.8, 21.7), (2100, 2100, 129): (21.6, 22.8), (2100, 2100, 161): (24.9, 23.2),
    (3000, 3000, 17): (17.6, 17.5), (3000, 3000, 97): (29.6, 18.3), (4000, 4000, 17): (21.5, 17.2),
    (5000, 5000, 3): (31.8, 23.2), (256, 8192, 65): (11.4, 13.7), (256, 8192, 161): (18.3, 14.2),
    (8192, 256, 33): (9.4, 13.5), (8192, 256, 193): (20.4, 15.1), (333, 777, 555): (45.3, 14.2),
    (411, 411, 411): (37.7, 14.0), (64, 1024, 1025): (66.5, 15.2), (100, 100, 6801): (429.0, 20.5),
    (4000, 17, 999): (59.6, 21.4), (1, 8192, 8193): (607.0, 106.0),
}


@pytest.mark.parametrize("shape", list(ODD_K))
def test_odd_k_picks_no_slower_path(rules, shape):
    generic, copies = ODD_K[shape]
    assert (generic, copies)[rules.pad(*shape)] <= 1.02 * min(generic, copies)


# grouped fp8: groups, rows each, N, K: transposed tile, persistent 128 x 256 tile
GROUPED = {
    (1, 100, 14336, 4096): (27.0, 29.7), (2, 100, 14336, 4096): (28.7, 30.1), (3, 100, 14336, 4096): (36.4, 34.8),
    (4, 100, 4096, 4096): (26.8, 28.3), (8, 16, 4096, 4096): (28.9, 28.9), (8, 128, 4096, 4096): (34.5, 31.5),
    (8, 190, 4096, 4096): (45.2, 34.3), (16, 130, 2048, 4096): (34.9, 32.6), (32, 129, 4096, 2048): (94.3, 76.9),
    (64, 16, 2048, 4096): (139.4, 101.4), (128, 130, 512, 512): (28.3, 24.3), (1, 100, 256, 4096): (24.4, 27.3),
    (3, 150, 256, 8192): (40.5, 46.3), (8, 64, 256, 7168): (36.7, 41.7), (8, 129, 128, 4096): (24.5, 28.1),
    (16, 129, 136, 1024): (14.6, 15.6), (16, 20, 512, 512): (15.2, 12.9), (16, 20, 1024, 2048): (18.4, 19.7),
    (8, 64, 2048, 4096): (26.4, 28.4), (2, 128, 16384, 2048): (21.9, 21.2), (4, 128, 8192, 1024): (17.7, 16.3),
    (5, 150, 7168, 2048): (37.2, 34.1), (6, 128, 5120, 1536): (20.9, 19.1), (12, 100, 4096, 4096): (41.2, 38.6),
}


@pytest.mark.parametrize("case", list(GROUPED))
def test_small_groups_pick_no_slower_tile(rules, case):
    G, rows, N, K = case
    trans, pers = GROUPED[case]
    assert (trans, pers)[rules.small_groups(G, G * rows, N, K)] <= 1.02 * min(trans, pers)


def test_small_groups_gpu_tests_reach_the_tile(rules):
    for G, M, N, K in [(8, 500, 264, 256), (9, 700, 2048, 640), (512, 32000, 128, 256), (4096, 4000, 8, 256),
                       (7, 1000, 520, 384), (64, 6400, 1000, 256), (10, 798, 1032, 640), (40, 4000, 2048, 512)]:
        assert rules.small_groups(G, M, N, K)
    assert not rules.small_groups(4, 4 * 192, 2048, 512)


# groups, rows each, N, K (skewed): caller's order, dealt over the XCDs
DEALT = {
    (64, 128, 2048, 4096): (142.3, 140.0), (128, 60, 2048, 4096): (226.4, 222.0), (128, 180, 2048, 2048): (168.7, 172.1),
    (64, 60, 2048, 4096): (117.7, 117.5), (64, 512, 2048, 4096): (286.0, 285.4), (16, 1000, 4096, 4096): (251.6, 255.0),
    (64, 128, 1024, 1024): (26.7, 29.2), (32, 128, 4096, 2048): (67.7, 68.6), (128, 128, 512, 512): (22.1, 24.3),
    (128, 128, 1024, 2048): (85.8, 90.0), (16, 128, 2048, 4096): (32.0, 35.5), (256, 128, 1024, 1024): (94.7, 102.4),
    (256, 128, 1024, 2048): (160.8, 167.2), (256, 60, 2048, 4096): (425.3, 437.7), (64, 20, 512, 512): (12.9, 14.5),
    (192, 20, 512, 512): (21.7, 26.3), (384, 20, 1024, 2048): (168.7, 187.0), (512, 20, 512, 512): (44.7, 69.3),
}


@pytest.mark.parametrize("case", list(DEALT))
def test_dealing_is_no_slower(rules, case):
    G, rows, N, K = case
    order, dealt = DEALT[case]
    assert (order, dealt)[rules.dealt(G, N, K)] <= 1.025 * min(order, dealt)
