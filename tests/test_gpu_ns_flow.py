"""Newton-Schulz in one launch (small and middling matrices): sides around its 64- and 128-tiles, every
combination of tile sizes, wide and tall outputs that 16-byte stores cannot take, more steps than one
launch holds, and calls on several streams at once, against the fp32 CPU oracle.

Tolerance: 1e-2 Frobenius-relative per five steps from 256 rows on, as for every other path.  With fewer
rows the rounding of the iterate to bf16 averages out less (1.2e-2 for 64 x 64, whatever computes it), so
there the bound is the error that rounding after every operation, as the reference does, makes on the same
input: this path rounds in a third of those places."""
import ctypes

import pytest
import torch

from flash_muon_amd import _lib, fast_newtonschulz, synthetic
from flash_muon_amd.muon import NS_COEFFS, NS_EPS
from oracle import oracle

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _check(got, G, steps):
    ref = oracle.newtonschulz(G, steps)
    tol = 1e-2 * -(-steps // 5) if min(G.shape) >= 256 else float(oracle.rel_fro(oracle.newtonschulz_eager_bf16(G, steps), ref))
    assert float(oracle.rel_fro(got, ref)) <= tol


# one 64-tile and its edges, X' on 64-tiles (at most 256 of them) and on 128-tiles, all on 128-tiles, both
# orientations; (rows, cols, batch)
@pytest.mark.parametrize("rows,cols,batch", [(64, 64, 1), (63, 65, 1), (65, 63, 2), (129, 1, 1), (127, 500, 3), (513, 512, 1),
                                             (384, 1537, 4), (1537, 384, 4), (512, 520, 8), (300, 700, 16), (700, 301, 16),
                                             (1024, 1024, 1), (1025, 1000, 1), (128, 4200, 2), (130, 130, 32)])
def test_shapes_against_oracle(rows, cols, batch):
    Gs = torch.stack([synthetic.gradient_like_bf16(rows, cols, min(8, rows, cols), 50 + i) for i in range(batch)])
    got = fast_newtonschulz(Gs.to(DEV) if batch > 1 else Gs[0].to(DEV), 5).cpu().view(Gs.shape)
    for i in {0, batch // 2, batch - 1}:
        _check(got[i], Gs[i], 5)


@pytest.mark.parametrize("steps", [1, 4, 6, 10, 11])
@pytest.mark.parametrize("rows,cols", [(200, 333), (320, 130)])
def test_step_counts_beyond_one_launch(rows, cols, steps):
    G = synthetic.gradient_like_bf16(rows, cols, 8, 9)
    _check(fast_newtonschulz(G.to(DEV), steps).cpu(), G, steps)


@pytest.mark.parametrize("rows,cols,batch", [(200, 333, 1), (512, 768, 8), (384, 384, 24)])
def test_same_bits_every_time_and_for_every_place_in_a_batch(rows, cols, batch):
    """What a workgroup draws and when is up to timing; the results are not."""
    G = synthetic.gradient_like_bf16(rows, cols, 8, 3).to(DEV)
    want = fast_newtonschulz(G, 5)
    for _ in range(3):
        got = fast_newtonschulz(G.expand(batch, rows, cols).contiguous(), 5)
        assert all(torch.equal(got[i], want) for i in range(batch))


def test_concurrent_streams():
    """Calls that share the GPU, each with workgroups that wait for each other inside a launch."""
    Gs = [synthetic.gradient_like_bf16(r, c, 8, 70 + i).to(DEV) for i, (r, c) in enumerate([(512, 512), (384, 1024), (1000, 640), (256, 256)])]
    want = [fast_newtonschulz(G, 5) for G in Gs]
    streams = [torch.cuda.Stream() for _ in Gs]
    torch.cuda.synchronize()
    got = []
    for _ in range(4):
        for G, s in zip(Gs, streams):
            with torch.cuda.stream(s):
                got.append(fast_newtonschulz(G, 5))
    torch.cuda.synchronize()
    for i, y in enumerate(got):
        assert torch.equal(y, want[i % len(Gs)])


# a K of up to 8192 in one launch, the next one in launches per product, which cut the first product along k; more matrices, up to 16384 and beyond
@pytest.mark.parametrize("rows,cols,batch", [(128, 8192, 1), (128, 8193, 1), (8200, 500, 1), (384, 9000, 8), (16400, 250, 8)])
def test_long_rows_on_both_sides_of_the_rule(rows, cols, batch):
    Gs = torch.stack([synthetic.gradient_like_bf16(rows, cols, 8, 30 + i % 2) for i in range(min(batch, 2))])
    got = fast_newtonschulz(Gs.to(DEV)[torch.arange(batch) % len(Gs)] if batch > 1 else Gs[0].to(DEV), 5).view(batch, rows, cols)
    for i in range(2, batch):
        assert torch.equal(got[i], got[i % 2])
    _check(got[0].cpu(), Gs[0], 5)


def test_the_scratch_of_launches_per_product_is_enough(lib):
    """Every step's iterate, in one launch, takes more memory than calls had to bring before: what fits them still runs, a byte less does not."""
    n, rows, cols = 12, 1152, 1500
    full, least = lib.fm_newtonschulz_batched_workspace_bytes(n, rows, cols), lib.fm_newtonschulz_batched_min_workspace_bytes(n, rows, cols)
    assert least < 0.8 * full
    assert lib.fm_newtonschulz_batched_min_workspace_bytes(1, 64, 64) == lib.fm_newtonschulz_batched_workspace_bytes(1, 64, 64)
    Gs = torch.stack([synthetic.gradient_like_bf16(rows, cols, 8, 7)] * n).to(DEV)
    outs = torch.empty_like(Gs)
    ws = torch.full((full,), 255, dtype=torch.uint8, device=DEV)
    ptrs = lambda t: (ctypes.c_void_p * n)(*[t[i].data_ptr() for i in range(n)])

    def call(ws_bytes):
        return lib.fm_newtonschulz_batched_bf16(ptrs(Gs), _lib.FM_BF16, n, rows, cols, cols, ptrs(outs), cols, 5, *NS_COEFFS, NS_EPS, ws.data_ptr(),
                                                ws_bytes, _lib.stream_ptr(Gs.device))

    for ws_bytes in (full, full - 1, least):
        outs.fill_(7.0)
        assert call(ws_bytes) == 0
        _check(outs[n - 1].cpu(), Gs[0].cpu(), 5)
    assert call(least - 1) == 6   # FM_ERR_WORKSPACE


def test_short_of_memory():
    """A stack that fitted with the smaller scratch still does (the allocator's limit set for the length of the test)."""
    G = synthetic.gradient_like_bf16(1920, 1920, 8, 5).to(DEV).expand(32, 1920, 1920).contiguous()
    want = fast_newtonschulz(G[:1], 5)
    torch.cuda.synchronize()
    torch.cuda.empty_cache()
    total = torch.cuda.get_device_properties(0).total_memory
    try:
        torch.cuda.set_per_process_memory_fraction((torch.cuda.memory_reserved() + 2.3e9) / total)
        got = fast_newtonschulz(G, 5)   # 0.24 GB of result and 1.7 GB of scratch, where the one launch takes 3.8
        torch.cuda.synchronize()
    finally:
        torch.cuda.set_per_process_memory_fraction(1.0)
    assert float(oracle.rel_fro(got[31].cpu(), want[0].float().cpu())) < 1e-2
