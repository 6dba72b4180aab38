"""Newton-Schulz in one launch (small and middling matrices): sides around its 64- and 128-tiles, every
combination of tile sizes, wide and tall outputs that 16-byte stores cannot take, more steps than one
launch holds, and calls on several streams at once, against the fp32 CPU oracle.

Tolerance: 1e-2 Frobenius-relative per five steps from 256 rows on, as for every other path.  With fewer
rows the rounding of the iterate to bf16 averages out less (1.2e-2 for 64 x 64, whatever computes it), so
there the bound is the error that rounding after every operation, as the reference does, makes on the same
input: this path rounds in a third of those places."""
import pytest
import torch

from flash_muon_amd import fast_newtonschulz, synthetic
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
