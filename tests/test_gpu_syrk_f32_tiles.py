"""fm_syrk_f32 at the edges of its schedule: sides around a 64-tile, k around a 32-stage, 16-byte and
4-byte copies, more tiles than one round, and the left-over tiles in equal pieces, with and without the
workspace their parts need.  Integer inputs: every sum is exact in fp32, so the product is too."""
import pytest
import torch

from flash_muon_amd import _lib, matmul_transpose, matmul_transpose_assign
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def syrk_f32_raw(X, with_ws):
    lib = _lib.load()
    M, K = X.shape
    Y = torch.empty(M, M, device=X.device)
    need = lib.fm_syrk_f32_workspace_bytes(M, K) if with_ws else 0
    ws = torch.full((max(need // 4, 1),), float("nan"), device=X.device)   # the parts need no initialisation
    st = lib.fm_syrk_f32(X.data_ptr(), X.stride(0), Y.data_ptr(), M, 1, M, K, ws.data_ptr() if need else None, need,
                         _lib.stream_ptr(X.device))
    _lib.check("fm_syrk_f32", st)
    return Y


def _ints(M, K, seed):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(-8, 9, (M, K), generator=g).float()


# (M, K): one tile and its neighbours; k remainders of 1, 4, 28 and 31; 253 tiles (kept whole), 528
# (one round and 16 tiles in pieces), 136 tiles with a long k (all in pieces, two tiles per piece), 1035 tiles
@pytest.mark.parametrize("M,K", [(63, 31), (64, 32), (65, 33), (128, 36), (191, 60), (1408, 64), (2048, 160),
                                 (2047, 513), (1024, 2048), (2880, 40)])
@pytest.mark.parametrize("with_ws", [True, False])
def test_integers_bit_exact(M, K, with_ws):
    X = _ints(M, K, M + K)
    want = oracle.xxt_int64(X).float()
    Y = syrk_f32_raw(X.to(DEV), with_ws)
    assert torch.equal(Y.cpu(), want)


@pytest.mark.parametrize("pitch,offset", [(68, 0), (67, 0), (68, 1)])
def test_pitch_and_alignment(pitch, offset):
    """Rows that allow 16-byte copies and rows that do not, in an output with an odd pitch."""
    M, K = 130, 64
    flat = torch.full((M * pitch + 8,), float("nan"))
    X = _ints(M, K, 7)
    flat[offset:offset + M * pitch].view(M, pitch)[:, :K] = X
    d = flat.to(DEV)[offset:offset + M * pitch].view(M, pitch)[:, :K]
    out = torch.zeros(M, M + 1, device=DEV)
    matmul_transpose_assign(d, out[:, :M])
    assert torch.equal(out[:, :M].cpu(), oracle.xxt_int64(X).float())
    assert (out[:, M] == 0).all()


def test_pieces_add_up_as_precisely_as_whole_tiles():
    """fp32 sums of K products: against fp64 both schedules stay under eps sqrt(K) (a random walk of K
    roundings of half a unit each, and a factor for the sums being of the size of the result)."""
    X = torch.randn(1024, 4096, generator=torch.Generator().manual_seed(1))
    assert _lib.load().fm_syrk_f32_workspace_bytes(1024, 4096) > 0
    ref = oracle.xxt(X, dtype=torch.float64)
    for Y in (matmul_transpose(X.to(DEV)), syrk_f32_raw(X.to(DEV), False)):
        assert float(oracle.rel_fro(Y.cpu(), ref)) < 2.0 ** -24 * 4096 ** 0.5
        assert torch.equal(Y, Y.T)
