"""The rules that choose kernels and schedules (csrc/fm_routes.h), built for the host and checked without a GPU."""
import ctypes
import os
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash_muon_amd", "csrc")
INT32_MAX = 2 ** 31 - 1

HOST = """
#include "fm_routes.h"
extern "C" {
long long scale_cast_rows_blocks(long long r, long long c) { return fm::scale_cast_rows_blocks(r, c); }
}
"""


@pytest.fixture(scope="module")
def routes(tmp_path_factory):
    d = tmp_path_factory.mktemp("routes")
    src, out = d / "routes.cpp", d / "routes.so"
    src.write_text(HOST)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-shared", "-fPIC", "-I", CSRC, str(src), "-o", str(out)], check=True)
    lib = ctypes.CDLL(str(out))
    lib.scale_cast_rows_blocks.restype = ctypes.c_longlong
    lib.scale_cast_rows_blocks.argtypes = [ctypes.c_longlong] * 2
    return lib


# the edge itself (chunks and a quarter of them up to 2^31 - 1), a matrix of 28.8 GB in bf16, and both sides of 2^31 chunks
@pytest.mark.parametrize("rows,cols", [(1, 8), (3, 1024), (1 << 20, 16384), (104857, 131072), (104858, 131072), (110000, 131072),
                                       (131071, 131072), (131072, 131072), (1 << 22, 1 << 20)])
def test_the_walk_over_rows_stays_below_two_to_the_31(routes, rows, cols):
    """scale_cast_rows_kernel counts in an int from block * 256 + thread in steps of the grid: the first value behind the last
    chunk still has to be representable for every thread, or a negative index passes the loop's test."""
    blocks = routes.scale_cast_rows_blocks(rows, cols)
    chunks = rows * cols // 8
    if blocks:
        stride = blocks * 256
        assert chunks <= 4 * stride and stride < chunks + 1024
        beyond = [t + (chunks - t + stride - 1) // stride * stride for t in (0, stride - 1, min(stride, chunks) - 1, (chunks - 1) % stride)]
        assert max(beyond) <= INT32_MAX
    else:   # what is left to the kernel of 64x64 tiles is only what would not fit
        assert chunks + chunks // 4 > INT32_MAX - 1024
