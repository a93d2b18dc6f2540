"""Host <-> device transfers of the runtime at the sizes where their route changes: a few bytes, rows that are no multiple of
16 bytes, the largest size a kernel copies (1 MiB), the largest that is staged (4 MiB), beyond it, and more uploads in a row than
the staging block holds.  Bytes come back exactly."""
import numpy as np
import pytest
import torch

from ttmlir_amd import datagen, runtime as rt

pytestmark = pytest.mark.gpu
DT, TL, ST = rt.DataType, rt.TensorLayout, rt.StorageType


@pytest.fixture(scope="module")
def device(dev):
    d = rt.open_mesh_device()
    yield d
    rt.close_mesh_device(d)


@pytest.mark.parametrize("tiled", [False, True])
@pytest.mark.parametrize("shape", [(1, 1), (3, 7), (512, 512), (513, 512), (1024, 1024), (1025, 1024), (3, 701, 1003)])
def test_float_round_trip_is_exact(device, shape, tiled):
    x = datagen.randn(shape, seed=3)
    lay = rt.Layout(ST.Device, TL.Tile if tiled else TL.RowMajor, DT.Float32)
    d = rt.to_layout(rt.from_torch(x), device, lay)
    assert torch.equal(rt.to_torch(rt.to_host(d, untilize=True)[0]), x)
    back = rt.to_layout(d, device, rt.Layout(ST.Host, TL.RowMajor, DT.BFloat16))   # two steps on the way back
    assert torch.equal(rt.to_torch(back), x.to(torch.bfloat16))


def test_more_uploads_than_the_staging_block_holds(device):
    xs = [datagen.randn((512, 1024), seed=i) for i in range(9)]      # 9 x 2 MiB through 8 MiB, none waited for
    lay = rt.Layout(ST.Device, TL.Tile, DT.Float32)
    ds = [rt.to_layout(rt.from_torch(x), device, lay) for x in xs]
    for x, d in zip(xs, ds):
        assert torch.equal(rt.to_torch(d), x)


def test_host_tensors_of_earlier_read_backs_keep_their_values(device):
    """Read-backs share a pool of host blocks: a block is not handed out again while its tensor lives."""
    lay = rt.Layout(ST.Device, TL.Tile, DT.BFloat16)
    xs = [datagen.randn((256, 320), seed=20 + i, dtype=torch.bfloat16) for i in range(6)]
    held = [rt.to_host(rt.to_layout(rt.from_torch(x), device, lay), untilize=True)[0] for x in xs[:4]]
    del held[1]
    held.append(rt.to_host(rt.to_layout(rt.from_torch(xs[4]), device, lay), untilize=True)[0])
    for x, h in zip([xs[0], xs[2], xs[3], xs[4]], held):
        assert torch.equal(rt.to_torch(h), x)
    assert np.array_equal(rt.to_numpy(held[0]), xs[0].view(torch.int16).numpy().view(np.uint16))


def test_the_routes_through_page_locked_memory_are_the_ones_that_run(device):
    """What the tests above compare would be the same bytes if the device were found not to reach page-locked memory."""
    x = datagen.randn((512, 1024), seed=1)
    lay = rt.Layout(ST.Device, TL.Tile, DT.Float32)
    rt.to_host(rt.to_layout(rt.from_torch(x), device, lay), untilize=True)    # a read-back waits: the staging block is empty
    rt.clear_stats()
    ds = [rt.to_layout(rt.from_torch(x), device, lay) for _ in range(5)]      # 5 x 2 MiB through 8 MiB
    assert rt.get_stat("StagingBlockReused") == 1
    for d in ds:
        assert torch.equal(rt.to_torch(d), x)
    assert rt.get_stat("HostPoolReadBack") == 5
