"""The rules that choose kernels and schedules (csrc/fm_routes.h), built for the host and checked without a GPU."""
import ctypes
import os
import subprocess

import pytest

import test_gpu_half_tail as half_tail

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "flash_muon_amd", "csrc")
INT32_MAX = 2 ** 31 - 1

HOST = """
#include "fm_routes.h"
extern "C" {
long long scale_cast_rows_blocks(long long r, long long c) { return fm::scale_cast_rows_blocks(r, c); }
int syrk_padded_pays(int M, int K, int rows, int aligned) { return fm::syrk_padded_pays(M, K, rows, aligned); }
int syrk_whole_in_place(int M, int K) { return fm::syrk_whole_in_place(M, K, 256); }
int syrk_copy_pays(int M, int K, int half) { return fm::syrk_copy_pays(M, K, half); }
int scale_cast_d_on_tiles(long long r, long long c) { return fm::scale_cast_d_on_tiles(r, c); }
int scale_cast_t_on_128(long long tiles) { return fm::scale_cast_t_on_128(tiles); }
int ns_flow_chosen(int batch, int m, int k) { return fm::ns_flow_chosen(batch, m, k); }
int half_tail_pays(int rem, int split, int nk) { return fm::half_tail_pays(rem, split, nk, 256); }
int slim_pays(int tiles, int nk) { return fm::slim_pays(tiles, nk, 256, fm::mid_parts(tiles, nk, 256), false); }
void ns_flow_launch(int steps, int i, int* out) { const fm::NsFlowLaunch n = fm::ns_flow_launch(steps, i); out[0] = n.first; out[1] = n.steps; out[2] = n.from; out[3] = n.turn; }
int ns_flow_slots() { return fm::kFlowSteps + 1; }
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


@pytest.mark.parametrize("side,on64,on128", [(768, 3.9, 4.3), (1024, 4.1, 4.3), (2048, 6.4, 5.4), (4096, 15.9, 13.0)])
def test_a_lone_transpose_is_cast_on_the_tiles_that_measured_faster(routes, side, on64, on128):
    assert bool(routes.scale_cast_t_on_128(ctypes.c_longlong((side // 128) ** 2))) == (on128 < on64)


@pytest.mark.parametrize("rows,cols,tiles,walk", [(1536, 1536, 4.1, 4.9), (2560, 2560, 6.4, 7.3), (2048, 5504, 9.2, 10.2), (4096, 4096, 12.4, 12.8),
                                                  (4096, 11008, 30.7, 28.1), (3000, 3000, 11.0, 8.5), (3, 1000000, 9.0, 5.3), (1000000, 8, 33.3, 7.6)])
def test_a_lone_cast_takes_the_kernel_that_measured_faster(routes, rows, cols, tiles, walk):
    assert bool(routes.scale_cast_d_on_tiles(ctypes.c_longlong(rows), ctypes.c_longlong(cols))) == (tiles < walk)


# (batch, M, K, us in one launch, us in launches per product), measured; the first ones are ordinary ratios
NS_TIMES = [(1, 1024, 4096, 212, 242), (2, 640, 2560, 156, 245), (6, 1408, 3872, 976, 1224), (16, 768, 3072, 672, 972), (4, 960, 3072, 441, 379),
            (1, 512, 8192, 221, 235), (1, 512, 10240, 306, 247), (1, 512, 16384, 398, 275), (1, 512, 65536, 1268, 629), (1, 512, 32768, 386, 274),
            (1, 128, 8192, 166, 179), (1, 128, 16384, 264, 198), (1, 1024, 5120, 314, 277), (1, 1024, 16384, 562, 445), (1, 768, 9216, 311, 265),
            (2, 512, 4096, 168, 228), (2, 512, 8192, 302, 263), (4, 256, 8192, 247, 262), (6, 256, 8192, 307, 267), (4, 512, 12288, 481, 631),
            (16, 640, 12288, 1959, 2383), (12, 384, 32768, 2112, 2281), (4, 576, 131072, 7547, 6641), (8, 256, 16384, 509, 531),
            (8, 512, 24576, 1682, 1587), (8, 128, 16384, 341, 293), (12, 1024, 6144, 1568, 1759), (4, 1024, 6144, 679, 822), (4, 1024, 8192, 921, 817),
            # sides of 11, 13 and 15 tiles of 128, from square to long; then 6, 9 and 10 of them
            (16, 1408, 7744, 4596, 4974), (16, 1408, 11264, 6681, 6581), (2, 1408, 2112, 364, 332), (3, 1408, 2816, 520, 440), (2, 1408, 1408, 249, 285),
            (12, 1664, 5488, 3428, 3757), (32, 1608, 3216, 5870, 6173), (28, 1608, 6432, 9348, 8948), (5, 1664, 1664, 605, 577), (12, 1664, 1664, 1253, 1821),
            (8, 1920, 3840, 2152, 2376), (24, 1856, 2784, 5090, 5280), (12, 1920, 5160, 4318, 4216), (32, 1920, 7680, 16558, 14446),
            (5, 1856, 5568, 1919, 2086), (7, 1920, 5760, 2766, 2531), (4, 1856, 7424, 1823, 1940), (4, 1856, 1856, 681, 674),
            (12, 744, 1992, 433, 571), (8, 768, 3072, 431, 559), (8, 696, 1864, 344, 321), (10, 768, 1760, 361, 352), (3, 1088, 1088, 212, 235),
            (3, 1088, 2176, 339, 307), (4, 1272, 3416, 586, 678), (4, 1160, 3112, 550, 517), (32, 1216, 4256, 4466, 4275),
            (3, 1024, 1280, 209, 240), (3, 1024, 1536, 272, 260), (4, 1024, 1024, 199, 234), (6, 960, 1440, 368, 339), (6, 1408, 11264, 2461, 2655)]


@pytest.mark.parametrize("batch,m,k,one,launches", NS_TIMES)
def test_one_launch_newtonschulz_where_it_measured_faster(routes, lib, batch, m, k, one, launches):
    assert bool(routes.ns_flow_chosen(batch, m, k)) == (one < launches)
    # one launch keeps every step's iterate and squares, in either orientation of the matrices
    if one < launches:
        need = lib.fm_newtonschulz_batched_workspace_bytes(batch, m, k)
        assert need >= batch * (6 * m * k + 10 * m * m) * 2
        assert need == lib.fm_newtonschulz_batched_workspace_bytes(batch, k, m)


# (M, K, us on 128x128 tiles - in place where the rows lie on lines, else behind a copy -, us padded to 256-tiles), measured
PADDED_TIMES = [(3664, 24072, 391, 340), (3748, 12000, 177.6, 187.1), (1956, 6000, 54.4, 55.5), (1960, 6896, 63.4, 58.5), (2043, 7496, 74, 67), (2468, 12000, 99.6, 115.9), (2560, 30416, 289, 223), (2468, 24000, 180, 191),
                (2212, 24000, 175.1, 172), (2200, 72576, 581, 416), (1000, 262144, 340, 497), (3200, 32768, 316.8, 405), (2980, 60000, 768, 531), (1956, 60000, 562, 298), (2980, 24000, 220, 319), (3936, 4000, 69.4, 77.4), (4056, 1248, 37.6, 42.8), (4000, 4000, 85.9, 77.7), (3000, 5000, 70.1, 75.7),
                (5280, 6000, 183, 167), (5792, 4000, 150, 193), (6048, 2000, 91, 122), (7776, 2000, 133, 161), (7580, 8040, 469, 429), (8096, 8040, 509, 453),
                (8008, 4000, 246, 263), (8008, 16000, 1102, 821), (10000, 8000, 887, 700), (10000, 4000, 402, 429), (11000, 16000, 2106, 1577), (12000, 8000, 1291, 959),
                (16008, 2000, 544, 646), (16008, 4000, 1159, 974), (16008, 8000, 2576, 1684), (20000, 2000, 782, 1017), (24000, 4000, 3036, 2152), (28000, 2000, 1727, 1920),
                (7552, 4096, 195, 253), (7552, 16384, 898, 781), (10112, 8192, 1007, 711), (12160, 2048, 276, 396), (12928, 8192, 1685, 1088), (16256, 8192, 2783, 1722)]


@pytest.mark.parametrize("M,K,tiles128,padded", PADDED_TIMES)
def test_large_products_of_ragged_sides_are_padded_where_it_measured_faster(routes, lib, M, K, tiles128, padded):
    pays = bool(routes.syrk_padded_pays(M, K, 0 if K % 64 == 0 else 1 if K % 32 == 0 else 2, M % 8 == 0))
    assert pays == (padded < tiles128)
    Mp, Kp = (M + 255) // 256 * 256, (K + 63) // 64 * 64
    if pays:   # room for both copies and the product's own scratch
        assert lib.fm_syrk_workspace_bytes(M, K) >= 2 * Mp * (Mp + Kp) + lib.fm_gemm_workspace_bytes(Mp, Mp)
    elif M % 128 == 0 and K % 64 == 0:   # whole tiles that are multiplied in place: the parts of left-over tiles at most
        assert lib.fm_syrk_workspace_bytes(M, K) <= (16 << 20) + 512


# (M, K, us on tiles of their own CU, us in place): odd numbers of whole 128-tiles
WHOLE_TIMES = [(128, 2048, 14.7, 12.0), (128, 65536, 34.5, 28.6), (384, 32768, 27.4, 23.5), (640, 2048, 16.1, 13.5), (640, 32768, 31.3, 28.1), (640, 85696, 53, 48.9), (1152, 1536, 13.8, 11.5),
               (1152, 4096, 23.5, 20.0), (1152, 32768, 57.0, 61.3), (1408, 1024, 11.5, 9.6), (1408, 2048, 16.9, 18.8), (1408, 4096, 27.4, 21.5), (1408, 16384, 47.8, 51.3),
               (1408, 32768, 80.1, 93.9), (1664, 1024, 11.7, 10.0), (1664, 2048, 17.2, 19.2), (1664, 3072, 23.0, 26.8), (1664, 4096, 27.4, 25.6), (1664, 12288, 50.9, 55.8),
               (1664, 32768, 108.5, 132.4), (1920, 1024, 12.0, 10.4), (1920, 2048, 17.5, 19.3), (1920, 3072, 23.4, 26.9), (1920, 6144, 39.9, 34.7), (1920, 32768, 125.3, 144.5),
               (2176, 2176, 20.7, 21.8), (2688, 2688, 26.3, 26.9), (2944, 2944, 46.7, 38.2), (8064, 1024, 114, 70)]


@pytest.mark.parametrize("M,K,apart,in_place", WHOLE_TIMES)
def test_odd_numbers_of_whole_tiles_are_multiplied_in_place_where_it_measured_faster(routes, M, K, apart, in_place):
    assert bool(routes.syrk_whole_in_place(M, K)) == (in_place < apart)


# (M, K, us with the 256-tiles left over cut along k, us with their halves in a launch of their own)
TAIL_TIMES = [(5888, 256, 40.9, 33.0), (5888, 1024, 63.3, 54.7), (6144, 256, 45.2, 34.1), (6144, 2048, 91.5, 86.4), (6400, 1024, 69.5, 57.2), (6400, 4096, 155.8, 148.5),
              (6400, 6144, 198.0, 207.0), (6400, 7168, 238.6, 241.6), (6656, 1024, 73.2, 58.0), (6656, 4096, 168.0, 151.4), (6656, 8192, 292.5, 276.0),
              (6912, 256, 54.6, 35.3), (6912, 4096, 173.6, 156.5)]


def _takes_halves(routes, tiles, nk):
    rem = tiles % 256
    return tiles >= 256 and 16 < rem <= 128 and nk > 1 and bool(routes.half_tail_pays(rem, min(256 // rem, nk, 16), nk))


@pytest.mark.parametrize("M,K,cut,halves", TAIL_TIMES)
def test_left_over_tiles_run_as_halves_where_it_measured_faster(routes, M, K, cut, halves):
    T = M // 256
    assert _takes_halves(routes, T * (T + 1) // 2, K // 64) == (halves < cut)


def test_what_the_gpu_tests_of_halves_run_on(routes):
    for M, K, _ in half_tail.HALVES:
        assert _takes_halves(routes, (M // 256) * (M // 256 + 1) // 2, K // 64), (M, K)
    for M, K, _ in half_tail.OTHERS:
        assert not _takes_halves(routes, (M // 256) * (M // 256 + 1) // 2, K // 64), (M, K)
    for M, K in half_tail.AXPBY_HALVES:
        assert _takes_halves(routes, (M // 256) * (K // 256), M // 64), (M, K)


# (M, K, us on whole 128-tiles or tiles cut along k, us on their halves): even numbers of tiles
SLIM_TIMES = [(1536, 1024, 11.1, 8.8), (1536, 4096, 27.8, 22.1), (1792, 2048, 17.4, 14.1), (1792, 4608, 30.7, 24.8), (1792, 6144, 39.7, 33.0),
              (512, 8192, 22.9, 33.9), (1024, 8192, 24.9, 35.5), (1536, 5120, 27.5, 29.8), (1536, 6144, 30.0, 32.2), (1536, 8192, 33.7, 38.0), (1664, 7680, 37.7, 40.5),
              (1792, 8128, 42.1, 43.8), (1920, 9216, 47.1, 48.1), (1792, 16384, 65.3, 70.3)]


@pytest.mark.parametrize("M,K,whole,halves", SLIM_TIMES)
def test_halves_of_tiles_are_taken_where_they_measured_faster(routes, M, K, whole, halves):
    T = M // 128
    assert bool(routes.slim_pays(T * (T + 1) // 2, K // 64)) == (halves < whole)


# (M, K, us in place, us behind a copy of X): rows that 16-byte copies can take and that lie on no lines
COPY_TIMES = [(3000, 5000, 75, 70), (7000, 2000, 129, 110), (2000, 2000, 23, 30), (4000, 1000, 33, 37), (1956, 12000, 93.6, 103.7), (2468, 12000, 99.6, 112.3),
              (2432, 9304, 92.4, 87.9), (2768, 9784, 106.9, 100.8), (1000, 65544, 106, 126), (1920, 65544, 349, 385), (3492, 6000, 117, 90), (4004, 4000, 88.2, 84.5), (5028, 6000, 183, 161)]


@pytest.mark.parametrize("M,K,in_place,copied", COPY_TIMES)
def test_rows_off_lines_are_copied_where_it_measured_faster(routes, M, K, in_place, copied):
    assert bool(routes.syrk_copy_pays(M, K, K % 32 == 0)) == (copied < in_place)


@pytest.mark.parametrize("name,value", [("FLASHMUON_KSPLIT", 2), ("FLASHMUON_NO_MID", 1), ("FLASHMUON_FAST_MIN_UNITS", 0), ("FLASHMUON_HALF", 0)])
def test_a_knob_leads_every_product_to_the_schedules_it_speaks_of(lib, knobs, name, value):
    """The workspaces are those of launches per product, and of copies padded to whole tiles with the product's own scratch."""
    per_product = lambda b, m, k: b * (4 * m * k + 2 * m * m) * 2
    assert lib.fm_newtonschulz_batched_workspace_bytes(12, 1152, 1152) > 12 * (6 + 10) * 1152 * 1152 * 2      # one launch
    knobs(name, value)
    need = lib.fm_newtonschulz_batched_workspace_bytes(12, 1152, 1152)                                          # padded to 1280
    assert per_product(12, 1280, 1280) < need < per_product(12, 1280, 1280) + lib.fm_gemm_workspace_bytes(1280, 1280) + (1 << 20)
    assert lib.fm_syrk_workspace_bytes(1000, 2000) >= 2 * 1024 * (2048 + 1024) + lib.fm_gemm_workspace_bytes(1024, 1024)
    assert lib.fm_syrk_workspace_bytes(1152, 4096) == lib.fm_gemm_workspace_bytes(1152, 1152)


@pytest.mark.parametrize("steps", range(1, 65))
def test_the_one_launch_iteration_stays_in_its_slots(routes, steps):
    """Every iterate that a launch reads or leaves behind lies in the workspace, each launch begins where the one before it
    left off, and what it leaves there is not one that it still reads."""
    done, at, i, out = 0, 0, 0, (ctypes.c_int * 4)()
    while done < steps:
        routes.ns_flow_launch(steps, i, out)
        first, n, slot, turn = out
        assert first == done and slot == at and n >= 1 and abs(turn) == 1
        done, at, i = done + n, at + n * turn, i + 1
        written = [slot + turn * s for s in range(1, n + (done < steps))]   # the last step of all writes the caller's output
        assert all(0 <= s < routes.ns_flow_slots() for s in [slot] + written)
        assert len(set([slot] + written)) == 1 + len(written)
    assert done == steps
