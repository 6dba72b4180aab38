"""128x128 tiles by workgroups in pairs (more whole tiles than compute units): the three products of a Newton-Schulz step
at sides of an odd number of tiles, one output or both, a stage of k and many, and batches; integer-valued inputs make every
comparison with the fp64 product bit-exact.  And Newton-Schulz at the edges of where it takes them, against the fp32
oracle (1e-2 Frobenius-relative per five steps, as for every other path)."""
import pytest
import torch

from flash_muon_amd import _lib, fast_newtonschulz, synthetic
from oracle import oracle
from tests import gpu_util

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ints(shape, seed, lo=-2, hi=2):
    g = torch.Generator().manual_seed(seed)
    return torch.randint(lo, hi + 1, shape, generator=g).float().bfloat16()


def _exact(x):
    return x.float().bfloat16()


@pytest.mark.parametrize("M,K", [(128, 33024), (1152, 3840), (1664, 2560), (384, 11008)])
def test_axpby(lib, M, K):   # 258, 270, 260 and 258 tiles
    P = _ints((M, M), 3 * M + K, -1, 1)
    X = _ints((M, K), 5 * M + K)
    d = torch.arange(M, dtype=torch.float32) % 3 - 1
    PX = P.double() @ X.double()
    want = _exact((2 + d.double())[:, None] * X.double() + PX)
    Xo, XoT = gpu_util.gemm_axpby(lib, P.to(DEV), X.to(DEV), 2.0, row_alpha=d.to(DEV))
    assert torch.equal(Xo.cpu(), want) and torch.equal(XoT.cpu(), want.T)
    want0 = _exact(2 * X.double() + PX)
    assert torch.equal(gpu_util.gemm_axpby(lib, P.to(DEV), X.to(DEV), 2.0, want_xt=False)[0].cpu(), want0)
    assert torch.equal(gpu_util.gemm_axpby(lib, P.to(DEV), X.to(DEV), 2.0, want_x=False)[1].cpu(), want0.T)


def test_poly(lib):   # 276 tiles
    M = 2944
    g = torch.Generator().manual_seed(M)
    A = torch.randint(-1, 2, (M, M), generator=g)
    A = (torch.triu(A) + torch.triu(A, 1).T).float().bfloat16()
    full = 2 * A.double() + 3 * (A.double() @ A.double())
    P, d = gpu_util.syrk_poly(lib, A.to(DEV), 2.0, 3.0, split_diag=True)
    assert torch.equal(d.cpu().double(), torch.diagonal(full))
    assert torch.equal(P.cpu(), _exact(full - torch.diag(torch.diagonal(full))))
    assert torch.equal(P, P.T)


def test_syrk_without_rows_on_lines(lib):
    """Rows that start between 128-byte lines keep the tiles of a whole multiple of 128 on this path."""
    M, K = 2944, 128
    buf = _ints((M, K + 8), 4)
    X = buf[:, :K]
    got = gpu_util.syrk(lib, buf.to(DEV)[:, :K])
    assert torch.equal(got.cpu(), _exact(X.double() @ X.double().T))


@pytest.mark.parametrize("rows,cols,batch", [(2300, 1100, 1), (2688, 2700, 1), (1409, 3300, 1), (650, 1700, 2), (1300, 1500, 4), (1900, 1921, 4),
                                             (1025, 3000, 4), (1500, 1536, 16)])
def test_newtonschulz_where_the_route_changes(rows, cols, batch):
    Gs = torch.stack([synthetic.gradient_like_bf16(rows, cols, 8, 90 + i % 2) for i in range(min(batch, 2))])
    Gd = Gs.to(DEV)[torch.arange(batch) % len(Gs)]
    got = fast_newtonschulz(Gd if batch > 1 else Gd[0], 5).view(batch, rows, cols)
    for i in range(2, batch):
        assert torch.equal(got[i], got[i % 2])
    assert float(oracle.rel_fro(got[0].cpu(), oracle.newtonschulz(Gs[0], 5))) <= 1e-2
