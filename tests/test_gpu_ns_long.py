"""Newton-Schulz steps on long matrices, as much about their accuracy as about their routes: every schedule that the products run on, padded
and transposed inputs, step counts, coefficients, and inputs whose rows are hard to tell apart.

Tolerance: no further from the iteration in 64 bits than steps one by one with the roundings of the kernels are: A, P without its
diagonal, and X to bf16, sums in fp32.  (The kernels themselves differ from that by the order of their sums, which turns some
roundings: a hundredth of the bound.)"""
import ctypes

import pytest
import torch

from flash_muon_amd import _lib, fast_newtonschulz
from flash_muon_amd.muon import NS_COEFFS, NS_EPS
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(rows, cols, dtype, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    u, v = torch.randn(rows, 32, generator=gen, device=DEV), torch.randn(32, cols, generator=gen, device=DEV)
    return (torch.randn(rows, cols, generator=gen, device=DEV) + 0.1 * u @ v).to(dtype)


def _one_by_one(X, steps, coeffs):
    a, b, c = coeffs
    X = X.bfloat16().float()
    for _ in range(steps):
        A = (X @ X.T).bfloat16().float()
        P = b * A + c * (A @ A)
        d = a + P.diagonal().clone()
        P = P.bfloat16().float().fill_diagonal_(0)
        X = (d[:, None] * X + P @ X).bfloat16().float()
    return X


def _check(got, G, steps, coeffs=NS_COEFFS):
    X = G.bfloat16().double()
    X = X.T.contiguous() if X.shape[0] > X.shape[1] else X
    got = got.double().T if got.shape[0] > got.shape[1] else got.double()
    X = X / (X.norm() + NS_EPS)
    want, by_one = X, _one_by_one(X.float(), steps, coeffs).double()
    for _ in range(steps):
        want = oracle.ns_step(want, coeffs)
    err, limit = (float((y - want).norm() / want.norm()) for y in (got, by_one))
    assert err <= 1.01 * limit and limit < 2e-2, (err, limit)


def _library_call(Gs, steps, coeffs=NS_COEFFS):
    """Through the C ABI with the least scratch, which keeps matrices of any size on launches per product."""
    lib = _lib.load()
    n, rows, cols = len(Gs), *Gs[0].shape
    outs = [torch.empty(rows, cols, dtype=torch.bfloat16, device=DEV) for _ in Gs]
    need = lib.fm_newtonschulz_batched_min_workspace_bytes(n, rows, cols)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    st = lib.fm_newtonschulz_batched_bf16((ctypes.c_void_p * n)(*[g.data_ptr() for g in Gs]), _lib.dtype_code(Gs[0].dtype), n, rows, cols, cols,
                                          (ctypes.c_void_p * n)(*[o.data_ptr() for o in outs]), cols, steps, *coeffs, NS_EPS,
                                          ws.data_ptr(), need, _lib.stream_ptr(Gs[0].device))
    _lib.check("fm_newtonschulz_batched_bf16", st)
    return outs


# from few 64x64 sub-tiles and 64x128 tiles over 128-tiles to rounds of 256-tiles with every way of dealing with their last ones
@pytest.mark.parametrize("rows,cols,batch", [(512, 1024, 1), (1664, 3328, 1), (640, 10240, 1), (1664, 3328, 4), (3072, 6144, 1), (4096, 8192, 1),
                                             (4096, 8192, 2), (2816, 5632, 5), (4096, 8192, 8), (8192, 16384, 1)])
def test_every_schedule_of_the_products(rows, cols, batch):
    Gs = [_inputs(rows, cols, torch.bfloat16, 7 + i) for i in range(batch)]
    outs = _library_call(Gs, 5)
    for i in {0, batch - 1}:
        _check(outs[i], Gs[i], 5)


# padded to 128- and 256-tiles, tall, fp32, into the output without a copy (5504 x 2048), K at and below twice M
@pytest.mark.parametrize("rows,cols,batch,dtype", [(2700, 1150, 1, torch.float32), (1150, 2700, 1, torch.float16), (5504, 2048, 3, torch.bfloat16),
                                                   (1600, 6401, 1, torch.float32), (1536, 3072, 8, torch.bfloat16), (1536, 3071, 1, torch.bfloat16),
                                                   (1664, 3328, 8, torch.bfloat16), (3200, 6400, 1, torch.bfloat16)])
def test_padded_and_transposed(rows, cols, batch, dtype):
    G = torch.stack([_inputs(rows, cols, dtype, 40 + i) for i in range(batch)])
    got = fast_newtonschulz(G if batch > 1 else G[0], 5).view(G.shape)
    for i in {0, batch - 1}:
        _check(got[i], G[i], 5)


# in one launch: whole and ragged tiles, tall, the fewest rows and columns, outputs that 16-byte stores cannot take
@pytest.mark.parametrize("rows,cols,batch,dtype", [(512, 1408, 16, torch.bfloat16), (3072, 768, 16, torch.float32), (1000, 2816, 8, torch.bfloat16),
                                                   (1921, 901, 12, torch.float16), (1408, 2820, 5, torch.bfloat16), (1150, 2301, 5, torch.float32)])
def test_in_one_launch(rows, cols, batch, dtype):
    G = torch.stack([_inputs(rows, cols, dtype, 60 + i) for i in range(batch)])
    got = fast_newtonschulz(G, 5)
    for i in {0, batch // 2, batch - 1}:
        _check(got[i], G[i], 5)
    again = fast_newtonschulz(G[:1].expand(batch, rows, cols).contiguous(), 5)
    assert all(torch.equal(again[i], got[0]) for i in range(batch))   # whatever workgroup draws what and when


@pytest.mark.parametrize("steps", [4, 5, 6, 7, 8, 10, 11, 16])
@pytest.mark.parametrize("batch", [1, 8])   # both in one launch per five steps
def test_step_counts(steps, batch):
    G = _inputs(1300, 2700, torch.bfloat16, 3)
    got = fast_newtonschulz(G.expand(batch, *G.shape).contiguous() if batch > 1 else G, steps).view(batch, *G.shape)
    _check(got[0], G, steps)
    assert all(torch.equal(got[0], g) for g in got)


def test_streams_at_once():
    Gs = [torch.stack([_inputs(r, c, torch.bfloat16, 80 + i) for i in range(b)]) for r, c, b in [(768, 2064, 8), (640, 1720, 16), (2816, 1024, 8)]]
    want = [fast_newtonschulz(G, 5) for G in Gs]
    streams = [torch.cuda.Stream() for _ in Gs]
    torch.cuda.synchronize()
    for _ in range(3):
        got = []
        for s, G in zip(streams, Gs):
            with torch.cuda.stream(s):
                got.append(fast_newtonschulz(G, 5))
        torch.cuda.synchronize()
        assert all(torch.equal(a, b) for a, b in zip(got, want))


@pytest.mark.parametrize("rows,cols,batch", [(768, 3072, 8), (1664, 4000, 1)])
def test_in_a_graph(rows, cols, batch):
    G = torch.stack([_inputs(rows, cols, torch.bfloat16, 90 + i) for i in range(batch)])
    for _ in range(2):
        want = fast_newtonschulz(G, 5)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        got = fast_newtonschulz(G, 5)
    for i in range(3):
        got.zero_()
        graph.replay()
        torch.cuda.synchronize()
        assert torch.equal(got, want)
        G.mul_(2.0)                          # the iterate, and with powers of two its bits, do not depend on the scale
        assert torch.equal(fast_newtonschulz(G, 5), want)


@pytest.mark.parametrize("coeffs", [(1.5, -0.5, 0.0), (1.875, -1.25, 0.375), (3.0, -3.2, 1.2), (4.0, -6.0, 3.0), (2.0, 0.0, 0.0)])
def test_other_coefficients(coeffs):
    G = _inputs(1664, 4000, torch.bfloat16, 4)
    _check(_library_call([G], 5, coeffs)[0], G, 5, coeffs)


def test_scales_of_the_input():
    """Rows over six decades: what is small beside the rest keeps its direction."""
    G = _inputs(1664, 4000, torch.float32, 5) * torch.logspace(0, -6, 1664, device=DEV)[:, None]
    got = fast_newtonschulz(G, 5)
    _check(got, G, 5)
    X = G.bfloat16().double()
    X = X / X.norm()
    for _ in range(5):
        X = oracle.ns_step(X)
    by_row = (got.double() - X).norm(dim=1) / X.norm(dim=1)
    by_one = (_one_by_one((G.bfloat16().float() / G.bfloat16().float().norm()), 5, NS_COEFFS).double() - X).norm(dim=1) / X.norm(dim=1)
    assert bool((by_row <= by_one.max()).all())


def _near(k, spread, rest):   # k rows that differ by `spread` of their size, beside others of size `rest`
    def make(gen, rows, cols):
        G = rest * torch.randn(rows, cols, generator=gen, device=DEV)
        G[:k] = torch.randn(1, cols, generator=gen, device=DEV) + spread * torch.randn(k, cols, generator=gen, device=DEV)
        return G
    return make


def _signs(gen, rows, cols):
    u, v = (torch.randn(*n, generator=gen, device=DEV).sign() for n in ((rows, 1), (1, cols)))
    return u * v + 1e-4 * torch.randn(rows, cols, generator=gen, device=DEV)


def _columns(decades):
    return lambda gen, rows, cols: torch.randn(rows, cols, generator=gen, device=DEV) * torch.logspace(0, -decades, cols, device=DEV)


HARD = {"4 alike, 1e-2": _near(4, 0.1, 1e-2), "4 alike, 1e-3": _near(4, 0.1, 1e-3), "3 alike, 1/3000": _near(3, 0.1, 1 / 3000),
        "16 alike, 1e-2": _near(16, 0.1, 1e-2), "8 equal, 1e-2": _near(8, 0.0, 1e-2), "64 equal, 1e-3": _near(64, 0.0, 1e-3),
        "128 equal, 1e-3": _near(128, 0.0, 1e-3), "signs": _signs, "columns 3": _columns(3), "columns 5": _columns(5)}


@pytest.mark.parametrize("kind", HARD)
@pytest.mark.parametrize("steps", [5, 8])
@pytest.mark.parametrize("rows,cols,batch", [(768, 3072, 8), (1664, 4000, 1)])   # in one launch, in launches per product
def test_rows_and_columns_that_amplify_roundings(kind, steps, rows, cols, batch):
    """Products of a few steps on M x M matrices alone, without X in between, lose 2 to 20 times as much here.  Bounds: the model
    itself with sums off by 2^-20 of their value, or in fp64, moves by up to 1.3 % (Frobenius) and a quarter (worst row); hence 2 % and 40 %.
    And no singular value comes near 1.2637, the root of p(s) = s beyond which the steps run away (exact ones end at 1.203)."""
    Gs = [HARD[kind](torch.Generator(device=DEV).manual_seed(i), rows, cols).bfloat16() for i in range(2)]
    got = fast_newtonschulz(torch.stack([Gs[i % 2] for i in range(batch)]) if batch > 1 else Gs[0], steps).view(batch, rows, cols)
    for i in range(min(batch, 2)):
        X = Gs[i].double()
        X = X / (X.norm() + NS_EPS)
        want, by_one = X, _one_by_one(X.float(), steps, NS_COEFFS).double()
        for _ in range(steps):
            want = oracle.ns_step(want)
        (err, row), (limit, row_limit) = ((float((y - want).norm() / want.norm()), float(((y - want).norm(dim=1) / want.norm(dim=1)).max()))
                                          for y in (got[i].double(), by_one))
        assert err <= 1.02 * limit and row <= 1.4 * row_limit, (err, limit, row, row_limit)
        Y, v = got[i].double(), torch.ones(rows, 1, dtype=torch.float64, device=DEV)
        for _ in range(60):   # the largest singular value, by powers of Y Y^T
            v = Y @ (Y.T @ (v / v.norm()))
        assert float(v.norm()) < 1.25 ** 2


def test_nan_and_zero():
    G = _inputs(1664, 4000, torch.bfloat16, 6)
    G[3, 5] = float("nan")
    assert bool(fast_newtonschulz(G, 5).isnan().all())
    assert float(fast_newtonschulz(torch.zeros_like(G), 5).float().abs().max()) == 0.0
