"""Tensors whose workgroups are more than one grid holds (2^32 lanes in a dimension): the chunk kernels of tilize and of block float
go out in several launches.  Tensors of tens of GiB, filled and compared in pieces."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.fixture()
def large(dev):
    yield dev
    torch.cuda.empty_cache()


def fill(t, seed):
    """Values that depend on the position in tensors of any size (torch's random fills stop at 2^31 elements)."""
    for i, p in enumerate(t.split(1 << 28)):
        p.copy_(torch.randint(1, 256, (p.numel(),), dtype=torch.uint8, device=t.device, generator=torch.Generator(device=t.device).manual_seed(seed + i)))


def test_tilize_and_untilize_of_a_row_of_2_31_elements(hip, large):
    """The row's last lanes lie beyond it, at columns that an int no longer holds."""
    cols = 2**31 - 77
    pc = -(-cols // 32) * 32
    x = torch.empty(cols, dtype=torch.uint8, device=large)
    fill(x, 1)
    t = torch.full((32 * pc,), 0x55, dtype=torch.uint8, device=large)
    hip.call("ttm_tilize", hip.ptr(x), hip.ptr(t), 1, 1, cols, 1, hip.current_stream())
    tiles, step = t.view(-1, 2, 2, 16, 16), 1 << 22      # tile, face row, face column, row, column
    for i in range(0, pc // 32, step):
        got, want = tiles[i:i + step], x[i * 32:(i + step) * 32]
        row = got[:, 0, :, 0, :].reshape(-1)
        assert torch.equal(row[:want.numel()], want) and not bool(row[want.numel():].any())
        assert not bool(got[:, 1].any()) and not bool(got[:, 0, :, 1:].any())
    back = torch.full((cols + 64,), 7, dtype=torch.uint8, device=large)
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(back), 1, 1, cols, 1, hip.current_stream())
    for got, want in zip(back[:cols].split(1 << 28), x.split(1 << 28)):
        assert torch.equal(got, want)
    assert bool((back[cols:] == 7).all())


def test_unpack_of_more_rows_than_a_grid_holds(hip, large):
    batch, rows, cols = 65535, 16400, 1
    matrix = -(-rows // 32) * 576
    packed = torch.empty(batch * matrix, dtype=torch.uint8, device=large)
    fill(packed, 2)
    out = torch.full((batch * rows + 64,), 7, dtype=torch.bfloat16, device=large)
    s = hip.current_stream()
    hip.call("ttm_bfp_unpack", hip.ptr(packed), hip.BFP4B, hip.ptr(out), hip.BF16, hip.ROW_MAJOR, batch, rows, cols, s)
    part = 8192
    for b in range(0, batch, part):
        n = min(part, batch - b)
        want = torch.empty(n * rows, dtype=torch.bfloat16, device=large)
        hip.call("ttm_bfp_unpack", hip.ptr(packed[b * matrix:]), hip.BFP4B, hip.ptr(want), hip.BF16, hip.ROW_MAJOR, n, rows, cols, s)
        assert torch.equal(out[b * rows:(b + n) * rows].view(torch.int16), want.view(torch.int16))
    assert bool((out[batch * rows:] == 7).all())


def test_unpack_of_a_row_of_2_31_elements(hip, large):
    cols, part = 2**31 - 77, 1 << 20   # tiles
    packed = torch.empty(-(-cols // 32) * 576, dtype=torch.uint8, device=large)
    fill(packed, 3)
    out = torch.full((cols + 64,), 7, dtype=torch.bfloat16, device=large)
    s = hip.current_stream()
    hip.call("ttm_bfp_unpack", hip.ptr(packed), hip.BFP4B, hip.ptr(out), hip.BF16, hip.ROW_MAJOR, 1, 1, cols, s)
    for tile in range(0, -(-cols // 32), part):
        n = min(part * 32, cols - tile * 32)
        want = torch.empty(n, dtype=torch.bfloat16, device=large)
        hip.call("ttm_bfp_unpack", hip.ptr(packed[tile * 576:]), hip.BFP4B, hip.ptr(want), hip.BF16, hip.ROW_MAJOR, 1, 1, n, s)
        assert torch.equal(out[tile * 32:tile * 32 + n].view(torch.int16), want.view(torch.int16))
    assert bool((out[cols:] == 7).all())
