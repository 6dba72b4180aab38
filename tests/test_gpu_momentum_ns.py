"""fm_momentum_newtonschulz_batched against the two calls it stands for: gradients, momenta and updates bit for bit, for
sizes with one unit per thread and several passes, tensors that 16-byte accesses cannot take, one-launch and per-product
iterations, and g or buf as what is orthogonalised; and what it refuses."""
import ctypes

import pytest
import torch

from flash_muon_amd import _lib
from flash_muon_amd.muon import NS_COEFFS, NS_EPS

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _ptrs(ts):
    return (ctypes.c_void_p * len(ts))(*[t.data_ptr() for t in ts])


def _tensors(batch, rows, cols, dtype, scale, seed, offset):
    g = torch.Generator().manual_seed(seed)
    out = []
    for _ in range(batch):
        flat = torch.zeros(rows * cols + 8, dtype=dtype, device=DEV)
        t = flat[offset:offset + rows * cols].view(rows, cols)
        t.copy_((scale * torch.randn(rows, cols, generator=g)).to(dtype))
        out.append(t)
    return out


def _fused(lib, gs, bufs, outs, nesterov, ws, steps=5):
    rows, cols = gs[0].shape
    return lib.fm_momentum_newtonschulz_batched(_ptrs(gs), _ptrs(bufs), _lib.dtype_code(gs[0].dtype), len(gs), rows, cols, 0.05, 0.95,
                                                nesterov, _ptrs(outs), cols, steps, *NS_COEFFS, NS_EPS, ws.data_ptr(), ws.numel(),
                                                _lib.stream_ptr(gs[0].device))


@pytest.mark.parametrize("batch,rows,cols,dtype,offset", [
    (3, 64, 100, torch.float32, 0), (2, 33, 77, torch.bfloat16, 0), (2, 96, 128, torch.float32, 1), (5, 300, 200, torch.float16, 0),
    (2, 1600, 700, torch.bfloat16, 0), (1, 1544, 1600, torch.float32, 0), (1, 2304, 2048, torch.bfloat16, 0), (2, 200, 12000, torch.float32, 0),
    (30, 1024, 1024, torch.float32, 0), (31, 1024, 1024, torch.float32, 0)])   # 120 MiB and more
@pytest.mark.parametrize("nesterov", [1, 0])
def test_same_bits_as_the_two_calls(lib, batch, rows, cols, dtype, offset, nesterov):
    gs = _tensors(batch, rows, cols, dtype, 1e-2, 1, offset)
    bufs = _tensors(batch, rows, cols, dtype, 1e-2, 2, offset)
    g2, b2 = [t.clone() if offset == 0 else t for t in gs], [t.clone() if offset == 0 else t for t in bufs]
    if offset:   # clones would be aligned
        g2, b2 = _tensors(batch, rows, cols, dtype, 1e-2, 1, offset), _tensors(batch, rows, cols, dtype, 1e-2, 2, offset)
    outs = [torch.empty(rows, cols, dtype=torch.bfloat16, device=DEV) for _ in gs]
    outs2 = [torch.empty_like(o) for o in outs]
    ws = torch.full((lib.fm_newtonschulz_batched_workspace_bytes(batch, rows, cols),), 255, dtype=torch.uint8, device=DEV)
    assert _fused(lib, gs, bufs, outs, nesterov, ws) == 0
    stream = _lib.stream_ptr(ws.device)
    dt = _lib.dtype_code(dtype)
    assert lib.fm_momentum_nesterov_batched(_ptrs(g2), _ptrs(b2), batch, dt, rows * cols, 0.05, 0.95, nesterov, stream) == 0
    assert lib.fm_newtonschulz_batched_bf16(_ptrs(g2 if nesterov else b2), dt, batch, rows, cols, cols, _ptrs(outs2), cols, 5, *NS_COEFFS,
                                            NS_EPS, ws.data_ptr(), ws.numel(), stream) == 0
    for x, y in zip(gs + bufs + outs, g2 + b2 + outs2):
        assert torch.equal(x, y)


def test_refuses_what_the_two_calls_refuse(lib):
    g, b = _tensors(1, 64, 64, torch.float32, 1.0, 1, 0), _tensors(1, 64, 64, torch.float32, 1.0, 2, 0)
    ws = torch.empty(lib.fm_newtonschulz_batched_workspace_bytes(1, 64, 64), dtype=torch.uint8, device=DEV)
    out = [torch.empty(64, 64, dtype=torch.bfloat16, device=DEV)]
    before = [t.clone() for t in g + b]
    assert _fused(lib, g, g, out, 1, ws) == _lib.FM_ERR_ALIAS
    assert _fused(lib, g, b, g, 1, ws) == _lib.FM_ERR_ALIAS
    assert _fused(lib, g, b, b, 1, ws) == _lib.FM_ERR_ALIAS
    assert _fused(lib, g, b, out, 1, ws[:256]) == 6          # FM_ERR_WORKSPACE
    assert _fused(lib, g, b, out, 1, ws, steps=-1) == 2      # FM_ERR_SHAPE
    # and the momentum update of a refused call has not been made
    for t, was in zip(g + b, before):
        assert torch.equal(t, was)
