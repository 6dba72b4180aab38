"""Newton-Schulz of sides of whole 128-tiles that is iterated on 256-tiles: the last product writes what exists of its
result straight into the caller's matrix.  Against the same call into rows that 16-byte stores cannot take, which goes
through a copy of the padded result: same bits, and nothing beside the rows is touched."""
import ctypes

import pytest
import torch

from flash_muon_amd import _lib
from flash_muon_amd.muon import NS_COEFFS, NS_EPS

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(lib, G, pitch):
    batch, rows, cols = G.shape
    out = torch.full((batch, rows + 1, pitch), 7.0, dtype=torch.bfloat16, device=DEV)
    ptr = lambda t: (ctypes.c_void_p * batch)(*[t[i].data_ptr() for i in range(batch)])
    ws = torch.full((lib.fm_newtonschulz_batched_workspace_bytes(batch, rows, cols),), 255, dtype=torch.uint8, device=DEV)
    assert lib.fm_newtonschulz_batched_bf16(ptr(G), _lib.dtype_code(G.dtype), batch, rows, cols, cols, ptr(out), pitch, 5, *NS_COEFFS, NS_EPS,
                                            ws.data_ptr(), ws.numel(), _lib.stream_ptr(G.device)) == 0
    assert bool((out[:, rows] == 7.0).all()) and bool((out[:, :rows, cols:] == 7.0).all())
    return out[:, :rows, :cols]


# whole 256-tiles in rounds and their parts or sub-tiles, half tiles, both sides padded or the long one, both orientations; of batches only the long
# one: 216 tiles of the last product, 264 (a round and 8, as sub-tiles), 288 (a round and 32, cut along k) and 168
@pytest.mark.parametrize("batch,rows,cols", [(1, 2944, 2944), (1, 3200, 4480), (1, 4480, 2944), (1, 2048, 2176), (1, 5504, 2048), (3, 2176, 2432),
                                             (6, 768, 2944), (6, 2688, 1024), (6, 1024, 2944), (6, 1024, 1664), (4, 2176, 2176)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_same_bits_as_through_a_copy(lib, knobs, batch, rows, cols, dtype):
    need = lib.fm_newtonschulz_batched_workspace_bytes(batch, rows, cols)
    knobs("FLASHMUON_NO_TICKETS", 0)   # as it is by itself; but a knob that is set leads to launches per product
    assert need == lib.fm_newtonschulz_batched_workspace_bytes(batch, rows, cols), "runs as one launch, which writes its result another way"
    knobs("FLASHMUON_NO_TICKETS", -1)
    g = torch.Generator(device=DEV).manual_seed(rows + cols)
    G = torch.randn(batch, rows, cols, generator=g, device=DEV).to(dtype)
    a = _run(lib, G, cols + 8)
    b = _run(lib, G, cols + 3)
    assert not bool((b == 7.0).any())
    assert torch.equal(a, b)


def test_general_path_writes_no_more(lib, knobs):
    knobs("FLASHMUON_NO_MID", 1)
    knobs("FLASHMUON_FAST_MIN_UNITS", 1 << 40)
    g = torch.Generator(device=DEV).manual_seed(1)
    G = torch.randn(1, 1536, 1664, generator=g, device=DEV).bfloat16()
    assert torch.equal(_run(lib, G, 1672), _run(lib, G, 1667))
