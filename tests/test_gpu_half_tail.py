"""Tiles left over after full rounds of 256-tiles that run as halves in a launch of their own: exact on integers, and
the bits of the other schedules but for the order of their sums."""
import pytest
import torch

from flash_muon_amd import _lib, matmul_transpose
from gpu_util import gemm_axpby

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ints(rows, cols, dtype, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-2, 3, (rows, cols), generator=gen, device=DEV).to(dtype)


# 20, 44, 69, 95 and 122 tiles left of a symmetric product, diagonal ones among them; 2, 5, 16 and 33 stages of 64
HALVES = [(M, K, dtype) for M in (5888, 6144, 6400, 6656, 6912)
          for K, dtype in [(128, torch.bfloat16), (320, torch.float16), (1024, torch.bfloat16), (2112, torch.bfloat16)] if (M, K) != (5888, 2112)]
# one stage, which cannot be cut along k; and what is cut
OTHERS = [(M, 64, torch.bfloat16) for M in (5888, 6144, 6656, 6912)] + [(5888, 2112, torch.bfloat16)]


@pytest.mark.parametrize("M,K,dtype", HALVES + OTHERS)
def test_symmetric_products_exact(M, K, dtype):
    X = _ints(M, K, dtype, M + K)
    Y = matmul_transpose(X)
    assert torch.equal(Y, Y.T)
    want = X.float() @ X.float().T          # integers below 2^24: exact in fp32, in any order
    assert torch.equal(Y, want.to(dtype))


# 20 and 104 tiles left of a product with an operand E and a transposed output, as halves; 17, cut along k
AXPBY_HALVES = [(512, 35328), (2304, 10240)]


@pytest.mark.parametrize("M,K", AXPBY_HALVES + [(3328, 5376)])
def test_axpby_exact(lib, M, K):
    P, X = _ints(M, M, torch.bfloat16, 1), _ints(M, K, torch.bfloat16, 2)
    Xo, XoT = gemm_axpby(lib, P, X, 3.0)
    want = (3.0 * X.float() + P.float() @ X.float()).bfloat16()
    assert torch.equal(Xo, want) and torch.equal(XoT, want.T)


def test_against_tiles_cut_along_k(lib):
    X = torch.randn(6656, 1024, generator=torch.Generator(device=DEV).manual_seed(3), device=DEV).bfloat16()
    Y = matmul_transpose(X)
    try:
        assert lib.fm_set_knob(_lib.FM_KNOB_HALF, 0) == 0 and lib.fm_set_knob(_lib.FM_KNOB_KSPLIT, 1) == 0
        whole = matmul_transpose(X)   # the tiles left over are cut along k
    finally:
        lib.fm_set_knob(_lib.FM_KNOB_HALF, -1)
        lib.fm_set_knob(_lib.FM_KNOB_KSPLIT, -1)
    # 256 whole tiles on both: rows of the first two bands
    assert torch.equal(Y[:2048, :2048], whole[:2048, :2048])
    assert float((Y.float() - whole.float()).norm() / whole.float().norm()) < 1e-3
