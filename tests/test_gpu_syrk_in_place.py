"""Symmetric products of 16-bit matrices that are read and written in place: sides around a 128-tile, the part of k
that a stage of 64 leaves, tiles in rounds, whole and in pieces along k, odd numbers of whole tiles, and inputs that are
copied first.  Integer inputs: every sum is exact in fp32 (and fp64), so the result is the exactly rounded one."""
import pytest
import torch

from flash_muon_amd import _lib, matmul_transpose_assign

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ints(M, K, seed, dtype):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-3, 4, (M, K), generator=g).to(dtype)


def _run(X, pitch_x, pitch_y, offset_y=0):
    """X in rows of pitch_x whose rest is NaN, into rows of pitch_y of an output that starts at an odd place."""
    M, K = X.shape
    x = torch.full((M, pitch_x), float("nan"), dtype=X.dtype, device=DEV)
    x[:, :K] = X.to(DEV)
    flat = torch.full((M * pitch_y + offset_y + 64,), 7.0, dtype=X.dtype, device=DEV)
    y = flat[offset_y:offset_y + M * pitch_y].view(M, pitch_y)
    matmul_transpose_assign(x[:, :K], y[:, :M])
    assert bool((y[:, M:] == 7.0).all()) and bool((flat[:offset_y] == 7.0).all()) and bool((flat[offset_y + M * pitch_y:] == 7.0).all())
    return y[:, :M].cpu()


# (M, K): sides one around whole tiles, tails of 8 and 56, K of one stage and a tail; 300 tiles, whole and (copied, in two
# pieces per CU) partly cut; 45 and 15 tiles in pieces, more than one round of tiles and a cut rest behind it; copied inputs (K
# odd, K below one stage, both sides padded); odd numbers of whole tiles, uncut and cut; 153 of them (the older path)
@pytest.mark.parametrize("M,K", [(1024, 72), (1023, 120), (1025, 128), (129, 520), (2999, 200), (4200, 136), (1100, 4088), (3000, 5000),
                                 (4100, 4104), (513, 8184), (700, 333), (1500, 57), (1, 65544), (1030, 64), (4000, 1504), (1408, 256),
                                 (4224, 128), (1152, 4096), (2176, 128)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_integers_bit_exact(M, K, dtype):
    X = _ints(M, K, M + K, dtype)
    want = (X.double() @ X.double().T).to(dtype)
    got = _run(X, K, M)
    assert torch.equal(got, want)


@pytest.mark.parametrize("pitch_x,pitch_y,offset_y", [(400, 777, 0), (408, 784, 8), (401, 776, 0), (400, 778, 3), (392, 777, 1)])
def test_pitches_and_alignment(pitch_x, pitch_y, offset_y):
    X = _ints(776, 392, 5, torch.bfloat16)
    want = (X.double() @ X.double().T).bfloat16()
    assert torch.equal(_run(X, pitch_x, pitch_y, offset_y), want)


def test_infinities_beside_the_rows():
    """What lies beyond a row's end takes no part, also where it is the next row's infinities."""
    X = torch.ones(600, 200, dtype=torch.bfloat16)
    X[:, :8] = 2.0
    X[300, 0] = float("inf")
    got = _run(X, 200, 600)
    want = (X.double() @ X.double().T).to(torch.bfloat16)
    assert torch.equal(got, want)


@pytest.mark.parametrize("M,K", [(5248, 12288), (5280, 6000), (1800, 56008)])
def test_what_outgrows_the_cache_is_padded(M, K):
    """An odd number of whole tiles, sides of neither, and few tile rows whose rows lie on no lines.  (Sums below 2^24: any fp32 product is exact.)"""
    X = _ints(M, K, 3, torch.bfloat16)
    x = X.to(DEV).float()
    want = (x @ x.T).bfloat16().cpu()
    assert torch.equal(_run(X, K, M), want)
    assert torch.equal(_run(X, K + 8, M + 5, 3), want)   # (rows off the lines)


def test_rows_that_can_be_read_are_read_in_place_where_there_is_no_room_for_a_copy(lib):
    """3000 x 4992 in rows off the lines is copied first, given the room; without it the same tiles and pieces run in place (the bits of the
    copied call; the general schedule adds in another order), and with no workspace at all the tiles stay whole."""
    M, K, pitch = 3000, 4992, 5000
    X = torch.randn(M, pitch, generator=torch.Generator().manual_seed(1)).bfloat16().to(DEV)
    full = lib.fm_syrk_workspace_bytes(M, K)
    ws = torch.full((full,), 255, dtype=torch.uint8, device=DEV)

    def call(ws_bytes):
        y = torch.empty(M, M, dtype=torch.bfloat16, device=DEV)
        _lib.check("fm_syrk_bf16", lib.fm_syrk_bf16(X.data_ptr(), pitch, y.data_ptr(), M, 1, M, K, ws.data_ptr(), ws_bytes, _lib.stream_ptr(X.device)))
        return y

    copied = call(full)
    assert torch.equal(call(16 << 20), copied)   # room for the parts alone
    y = torch.empty(M, M, dtype=torch.bfloat16, device=DEV)
    _lib.check("fm_syrk_bf16_static", lib.fm_syrk_bf16_static(X.data_ptr(), pitch, y.data_ptr(), M, 1, M, K, _lib.stream_ptr(X.device)))
    assert torch.equal(y, copied)
    whole = call(0)
    assert torch.equal(whole, whole.T)
    # tiles that nothing cuts: the first 4 rows of tiles, in the order they are kept whole in
    assert torch.equal(whole[:512, :512], copied[:512, :512])
    assert float((whole.float() - copied.float()).norm() / copied.float().norm()) < 1e-3


def test_padded_copies_that_find_no_memory():
    """5248 x 12288 is padded, in 0.25 GB of scratch; where that cannot be had the product runs in place, as it did with 16 MiB."""
    _lib.release_workspaces()
    X = _ints(5248, 12288, 4, torch.bfloat16).to(DEV)
    x = X.float()
    want = (x @ x.T).bfloat16()
    y = torch.empty_like(want)
    del x
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 64e6) / total)
        matmul_transpose_assign(X, y)
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert torch.equal(y, want)
