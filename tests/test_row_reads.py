"""Which softmax tensors are read through the caches (csrc/kernels/row_reads.hpp), on the CPU."""
import ctypes
import os
import subprocess

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SOURCE = """
#include "row_reads.hpp"
extern "C" int past(int64_t rows, int64_t row_bytes) { return mtrt_dev::softmax_reads_past(rows, row_bytes); }
"""


def test_rows_that_share_lines_go_through_the_caches_from_20_to_80_mib(tmp_path):
    src, lib = tmp_path / "reads.cpp", tmp_path / "reads.so"
    src.write_text(SOURCE)
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-I", os.path.join(ROOT, "tensorrt-incubator_amd", "csrc", "kernels"), "-o", str(lib), str(src)],
                   check=True)
    past = ctypes.CDLL(str(lib)).past
    past.argtypes = [ctypes.c_int64, ctypes.c_int64]
    low, high = 20 << 20, 80 << 20
    for row_bytes in (2, 20, 64, 100, 192, 1000, 2002, 3000, 3008, 4112, 18002, 49016, 100000):
        for rows, expected in ((1, True), (low // row_bytes, True), (low // row_bytes + 1, False), (high // row_bytes, False), (high // row_bytes + 1, True),
                               ((1 << 41) // row_bytes, True)):
            assert past(rows, row_bytes) == expected, (rows, row_bytes)
    for row_bytes in (128, 256, 1920, 2048, 3968, 8192, 24064, 65536):             # whole lines
        assert all(past(size // row_bytes, row_bytes) for size in (1 << 20, low + row_bytes, 50 << 20, high, 1 << 40))
