"""Tilize / untilize of shapes the ragged strip kernel takes (rows that are no multiple of 16 bytes, row ends inside a strip, one
tile column past a strip, several matrices, a last strip of one column), on buffers that start at any element: bytes and zero padding
against the oracle, and nothing written around the destination."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("dtype", [np.uint32, np.uint16, np.uint8])
@pytest.mark.parametrize("batch,rows,cols,shift", [(3, 1000, 3001, 0), (1, 2050, 4097, 1), (2, 800, 2047, 3), (64, 33, 1023, 0), (1, 8192, 513, 1),
                                                  (1, 4096, 4000, 0), (5, 24, 7001, 5)])
def test_strips(hip, dev, orc, dtype, batch, rows, cols, shift):
    rng = np.random.default_rng(rows + cols)
    n, e = batch * rows * cols, np.dtype(dtype).itemsize
    x = rng.integers(0, 256, n * e, dtype=np.uint8).view(dtype)
    tdt = {4: torch.int32, 2: torch.int16, 1: torch.uint8}[e]
    as_t = lambda a: torch.from_numpy(a.view({4: np.int32, 2: np.int16, 1: np.uint8}[e]))
    pad = 64
    src = torch.zeros(n + 2 * pad, dtype=tdt, device=dev)
    src[pad + shift:pad + shift + n] = as_t(x).to(dev)
    pr, pc = (rows + 31) // 32 * 32, (cols + 31) // 32 * 32
    tiles = torch.full((batch * pr * pc,), 7, dtype=tdt, device=dev)
    s = hip.current_stream()
    hip.call("ttm_tilize", hip.ptr(src[pad + shift:]), hip.ptr(tiles), batch, rows, cols, e, s)
    want = np.concatenate([orc.tilize(m).reshape(-1) for m in x.reshape(batch, rows, cols)])
    assert np.array_equal(tiles.cpu().numpy().view(dtype), want)
    back = torch.full((n + 2 * pad,), 5, dtype=tdt, device=dev)
    hip.call("ttm_untilize", hip.ptr(tiles), hip.ptr(back[pad + shift:]), batch, rows, cols, e, s)
    got = back.cpu().numpy().view(dtype)
    assert np.array_equal(got[pad + shift:pad + shift + n], x)
    assert (got[:pad + shift] == 5).all() and (got[pad + shift + n:] == 5).all()
