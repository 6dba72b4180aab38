"""Halves of 128x128 tiles, at most one a CU: exact on integers for every write-out it has, diagonal tiles as two items and as one, 1 to 40
stages (around the six of its ring), and an operand E; batches of all three products of a Newton-Schulz step."""
import pytest
import torch

from flash_muon_amd import matmul_transpose
from flash_muon_amd.muon import NS_EPS
from gpu_util import gemm_axpby, syrk_poly
from test_gpu_ns_long import _library_call, _one_by_one

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ints(rows, cols, dtype, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    return torch.randint(-2, 3, (rows, cols), generator=gen, device=DEV).to(dtype)


# 1536 and 1920: two items per diagonal tile; 2048: one; a ring of six stages: fewer, as many, one and a round more
@pytest.mark.parametrize("M", [1536, 1792, 1920, 2048])
@pytest.mark.parametrize("K", [64, 128, 320, 384, 448, 1024, 2560])
def test_symmetric_products_exact(M, K):
    for dtype in (torch.bfloat16, torch.float16):
        X = _ints(M, K, dtype, M + K)
        Y = matmul_transpose(X)
        assert torch.equal(Y, (X.float() @ X.float().T).to(dtype))
        assert torch.equal(Y, Y.T)


def test_symmetric_bits_on_gaussian_input():
    for M in (1792, 2048):
        X = torch.randn(M, 2048, generator=torch.Generator(device=DEV).manual_seed(M), device=DEV).bfloat16()
        Y = matmul_transpose(X)
        want = X.double() @ X.double().T
        assert torch.equal(Y, Y.T)
        # fp32 sums (1e-6) and one rounding to 8 bits, up to half a unit of the last, which is 2^-8 of the value at most: evenly
        # spread errors are 2^-8 / sqrt(3) of it on the root mean square at most
        assert float((Y.double() - want).norm() / want.norm()) <= 2.0 ** -8 / 3 ** 0.5


@pytest.mark.parametrize("M", [1536, 1664, 2048])
def test_poly_exact(lib, M):
    """b A + c A A with the diagonal in fp32, or stored."""
    A = _ints(M, M, torch.float32, 5)
    A = (A + A.T).bfloat16()
    want = 2.0 * A.float() - 3.0 * (A.float() @ A.float())
    P = syrk_poly(lib, A, 2.0, -3.0)
    assert torch.equal(P, want.bfloat16())
    P, d = syrk_poly(lib, A, 2.0, -3.0, split_diag=True)
    assert torch.equal(d, want.diagonal())
    assert torch.equal(P, want.bfloat16().fill_diagonal_(0))


# 8 x 16 and 11 x 11 tiles; either output alone
@pytest.mark.parametrize("M,K,x,xt", [(1024, 2048, True, True), (1408, 1408, True, False), (1408, 1408, False, True), (128, 384, True, True)])
def test_axpby_exact(lib, M, K, x, xt):
    P, X = _ints(M, M, torch.bfloat16, 1), _ints(M, K, torch.bfloat16, 2)
    ra = torch.arange(M, device=DEV, dtype=torch.float32) % 5
    Xo, XoT = gemm_axpby(lib, P, X, 3.0, want_x=x, want_xt=xt, row_alpha=ra)
    want = ((3.0 + ra)[:, None] * X.float() + P.float() @ X.float()).bfloat16()
    assert not x or torch.equal(Xo, want)
    assert not xt or torch.equal(XoT, want.T)


# A and P of 4 matrices of 8 tile rows and 2 of 11: 256 and 242 items, a diagonal tile as one; of 3 of 7: 168, as two; X' of 2 of 5 x 12: 240
@pytest.mark.parametrize("batch,M,K", [(4, 1024, 2816), (2, 1408, 2816), (3, 896, 1792), (2, 640, 1536)])
@pytest.mark.parametrize("tall", [False, True])
def test_batches(batch, M, K, tall):
    """One step, in launches per product, of matrices that differ: each against the same roundings in fp32, whose sums have another order (that turns
    less than one rounding in a hundred, by a unit of 2^-8 at most: 8e-4 on the root mean square); and of equal ones, whose bits are equal."""
    Gs = [torch.randn(M, K, generator=torch.Generator(device=DEV).manual_seed(i), device=DEV).bfloat16() for i in range(batch)]
    put = (lambda G: G.T.contiguous()) if tall else (lambda G: G)
    for G, out in zip(Gs, _library_call([put(G) for G in Gs], 1)):
        X = G.float()
        want = _one_by_one(X / (X.norm() + NS_EPS), 1, (3.4445, -4.7750, 2.0315))
        got = (out.T if tall else out).float()
        assert float((got - want).norm() / want.norm()) < 8e-4
    outs = _library_call([put(Gs[-1])] * batch, 1)
    assert all(torch.equal(outs[0], o) for o in outs) and torch.equal(outs[0], _library_call([put(G) for G in Gs], 1)[-1])
