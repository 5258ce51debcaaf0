"""The row-wise quantiser's rule for 1024 threads per row, on the CPU: taken from
tx_op_quant.cpp, compiled by itself, and held to launches timed both ways on
one MI355X (microseconds; 256 CUs).  It may not pick a side that is more than
2% slower.
"""
import ctypes
import os
import re
import shutil
import subprocess

import pytest

SRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "triton-ext_amd", "csrc", "host",
                   "tx_op_quant.cpp")
# fp32, rows, K: 256 threads, 1024 threads
MEASURED = {
    (0, 1, 4096): (2.91, 2.93), (0, 1, 8192): (3.50, 3.35), (0, 1, 16384): (6.11, 4.01), (0, 16, 2056): (3.11, 3.25),
    (0, 16, 6144): (3.47, 3.36), (0, 16, 14336): (5.93, 3.98), (0, 128, 3072): (3.24, 3.36), (0, 200, 4096): (3.33, 3.46),
    (0, 256, 4096): (3.33, 3.50), (0, 256, 8192): (4.06, 3.95), (0, 256, 8200): (5.01, 4.08), (0, 384, 2056): (3.38, 4.33),
    (0, 384, 8192): (4.55, 5.24), (0, 384, 10240): (5.95, 5.61), (0, 511, 4096): (3.71, 4.61), (0, 511, 8192): (4.73, 5.41),
    (0, 511, 8200): (5.79, 5.68), (0, 600, 8200): (6.64, 7.47), (0, 600, 12288): (7.92, 8.28), (0, 600, 16384): (9.62, 9.61),
    (0, 1024, 10240): (8.88, 9.81), (0, 1024, 14336): (12.16, 11.66), (0, 2048, 9216): (15.7, 17.2), (0, 2048, 12288): (20.5, 19.0),
    (0, 4096, 8200): (26.0, 30.9), (0, 4096, 10240): (31.0, 31.5), (0, 4096, 11264): (34.3, 33.9), (0, 4096, 14336): (43.4, 37.3),
    (0, 8192, 9216): (52.8, 55.8), (0, 8192, 16384): (103.8, 83.3),
    (1, 1, 2056): (3.16, 2.79), (1, 1, 8192): (5.14, 3.56), (1, 16, 1032): (3.12, 3.07), (1, 16, 4096): (3.86, 3.35),
    (1, 200, 1032): (3.20, 3.27), (1, 256, 2056): (3.60, 3.37), (1, 256, 16384): (11.1, 5.68), (1, 384, 1032): (3.30, 3.99),
    (1, 384, 4096): (4.08, 4.47), (1, 511, 2056): (3.73, 4.27), (1, 511, 6144): (4.99, 4.89), (1, 511, 8192): (5.86, 5.58),
    (1, 600, 8200): (6.89, 7.57), (1, 600, 9216): (7.70, 8.05), (1, 600, 10240): (9.60, 8.46), (1, 1024, 8200): (10.77, 10.75),
    (1, 1024, 10240): (14.8, 13.5), (1, 4096, 8200): (43.5, 35.9), (1, 4096, 16384): (91.7, 69.4),
}


@pytest.fixture(scope="module")
def rule(tmp_path_factory):
    if not shutil.which("g++"):
        pytest.skip("needs g++")
    with open(SRC) as f:
        fn = re.search(r"^bool quant_row_wide\(.*?^}", f.read(), re.M | re.S)[0]
    d = tmp_path_factory.mktemp("rule")
    cpp, so = str(d / "rule.cpp"), str(d / "rule.so")
    with open(cpp, "w") as f:
        f.write("#include <cstdint>\n" + fn + '\nextern "C" int wide(bool f32, int64_t rows, int64_t K) '
                "{ return quant_row_wide(f32, rows, K, 256); }\n")
    subprocess.run(["g++", "-O1", "-std=c++17", "-shared", "-fPIC", cpp, "-o", so], check=True)
    lib = ctypes.CDLL(so).wide
    lib.argtypes = [ctypes.c_bool, ctypes.c_int64, ctypes.c_int64]
    return lambda *a: bool(lib(*a))


@pytest.mark.parametrize("case", list(MEASURED))
def test_picks_no_slower_form(rule, case):
    narrow, wide = MEASURED[case]
    assert (narrow, wide)[rule(*case)] <= 1.02 * min(narrow, wide)
    assert not rule(case[0], case[1], 16385)  # more than 1024 threads hold
