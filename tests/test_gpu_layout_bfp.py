"""GPU parity: tilize / untilize and bfp8_b / bfp4_b pack / unpack through the C ABI, bit exact
against the CPU oracle on the same seeded inputs, plus size-independent properties at the
full benchmark size (8192 x 8192)."""
import numpy as np
import pytest
import torch

from ttmlir_amd import datagen

pytestmark = pytest.mark.gpu

NP2T = {np.dtype(np.float32): torch.float32, np.dtype(np.uint16): torch.int16, np.dtype(np.uint8): torch.uint8,
        np.dtype(np.int32): torch.int32}


@pytest.fixture(autouse=True)
def by_the_rule(request):
    """Every test leaves the kernel choice to the rules, whatever it sets and however it ends."""
    h = request.getfixturevalue("hip") if "hip" in request.fixturenames else None
    yield
    if h is not None:
        for option in ("tilize_variant", "untilize_variant", "pack_variant", "unpack_variant"):
            h.set_option(option, 0)


def to_dev(x, dev):
    return torch.from_numpy(x.view(np.int16) if x.dtype == np.uint16 else x).to(dev)


def run_tilize(hip, dev, x, variant=0, untilize_shape=None):
    b, r, c = x.shape[:-2], x.shape[-2], x.shape[-1]
    batch = int(np.prod(b, dtype=np.int64))
    pr, pc = (r + 31) // 32 * 32, (c + 31) // 32 * 32
    xd = to_dev(x, dev)
    out = torch.full((batch * pr * pc,), 0x55, dtype=xd.dtype, device=dev)
    hip.set_option("tilize_variant", variant)
    hip.call("ttm_tilize", hip.ptr(xd), hip.ptr(out), batch, r, c, x.dtype.itemsize, hip.current_stream())
    torch.cuda.synchronize()
    return out


@pytest.mark.parametrize("variant", [0, 1, 2])
@pytest.mark.parametrize("shape,dtype", [((256, 512), np.uint16), ((512, 256), np.uint16), ((64, 128), np.float32),
                                         ((3, 64, 256), np.float32), ((2, 2, 32, 32), np.uint8),
                                         ((96, 1536), np.uint8), ((1024, 1024), np.float32)])
def test_tilize_untilize_bit_exact(hip, dev, orc, shape, dtype, variant):
    rng = np.random.default_rng(0)
    x = rng.integers(0, 2 ** (8 * np.dtype(dtype).itemsize) - 1, size=shape, dtype=np.uint64).astype(
        np.uint32).astype(dtype) if dtype != np.float32 else rng.standard_normal(shape).astype(np.float32)
    t = run_tilize(hip, dev, x, variant)
    want = orc.tilize(x)
    got = t.cpu().numpy().view(x.dtype)
    assert np.array_equal(got.view(np.uint8), want.view(np.uint8))
    # and back
    back = torch.empty_like(to_dev(x, dev))
    hip.set_option("untilize_variant", variant)
    batch = int(np.prod(shape[:-2], dtype=np.int64))
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(back), batch, shape[-2], shape[-1], x.dtype.itemsize,
             hip.current_stream())
    torch.cuda.synchronize()
    assert np.array_equal(back.cpu().numpy().view(x.dtype).view(np.uint8), x.view(np.uint8))


@pytest.mark.parametrize("dtype", [np.float32, np.uint16, np.uint8])
@pytest.mark.parametrize("shape", [(1, 1), (5, 7), (33, 31), (3, 17, 40), (1, 100), (40, 4096), (3, 500, 1000), (2, 70, 1002), (65, 33),
                                   (2, 2, 31, 64)])
def test_tilize_ragged_zero_padded(hip, dev, orc, shape, dtype):
    """Shapes that are not multiples of 32 in 4-, 2- and 1-byte elements: rows whose row-major start is 16-byte aligned in
    every row, in every other row, in none; batches; the padding of the tiles is zero, untilize leaves nothing outside the
    row-major tensor (the buffer is longer than it and must keep its fill)."""
    rng = np.random.default_rng(1)
    x = rng.standard_normal(shape).astype(np.float32) if dtype == np.float32 else rng.integers(1, 250, shape).astype(dtype)
    t = run_tilize(hip, dev, x)
    assert np.array_equal(t.cpu().numpy().view(dtype), orc.tilize(x).view(dtype).reshape(-1))
    n = int(np.prod(shape))
    back = torch.full((n + 64,), 7, dtype=t.dtype, device=dev)
    b, r, c = orc._split3(shape)
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(back), b, r, c, x.dtype.itemsize, hip.current_stream())
    torch.cuda.synchronize()
    got = back.cpu().numpy().view(dtype)
    assert np.array_equal(got[:n].reshape(shape), x)
    assert np.all(got[n:] == np.asarray(7, dtype=back.cpu().numpy().dtype).view(dtype))


@pytest.mark.parametrize("dtype", [np.float32, np.uint16, np.uint8])
@pytest.mark.parametrize("shape,offset", [((70, 1002), 1), ((3, 33, 129), 3), ((5, 3, 8), 1), ((40, 4, 17), 5), ((1, 1), 1), ((2, 65, 515), 7),
                                          ((2, 1000, 1003), 1), ((2, 1000, 1027), 3),   # bf16: 4 MiB, and beyond it
                                          ((2, 70, 283), 1), ((2, 70, 570), 3), ((3, 40, 1140), 1)])   # one and two wavefronts side by side
@pytest.mark.parametrize("variant", [0, 2])
def test_tilize_untilize_at_any_element(hip, dev, orc, shape, dtype, offset, variant):
    """Chunk by chunk, and untilized by strips: the row-major side starts at any element of its buffer and nothing in front of it or
    behind it is written; rows narrower than a wavefront's access, matrices shorter than a workgroup's."""
    rng = np.random.default_rng(2)
    x = rng.standard_normal(shape).astype(np.float32) if dtype == np.float32 else rng.integers(1, 250, shape).astype(dtype)
    n = x.size
    b, r, c = orc._split3(shape)
    hip.set_option("tilize_variant", variant)
    hip.set_option("untilize_variant", variant)
    buf = torch.full((n + 64,), 7, dtype=NP2T[np.dtype(dtype)], device=dev)
    rm = buf[offset:offset + n]
    rm.copy_(to_dev(x, dev).reshape(-1))
    t = torch.full((b * (-(-r // 32) * 32) * (-(-c // 32) * 32),), 0x55, dtype=buf.dtype, device=dev)
    hip.call("ttm_tilize", hip.ptr(rm), hip.ptr(t), b, r, c, x.dtype.itemsize, hip.current_stream())
    assert np.array_equal(t.cpu().numpy().view(dtype), orc.tilize(x).view(dtype).reshape(-1))
    rm.fill_(9)
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(rm), b, r, c, x.dtype.itemsize, hip.current_stream())
    got = buf.cpu().numpy().view(dtype)
    seven = np.full(1, 7, dtype=buf.cpu().numpy().dtype).view(dtype)[0]
    assert np.array_equal(got[offset:offset + n].reshape(shape), x)
    assert np.all(got[:offset] == seven) and np.all(got[offset + n:] == seven)


def test_untilize_by_strips_of_more_matrices_than_a_grid_has_rows(hip, dev):
    batch, r, c = 65600, 3, 5
    t = torch.randint(0, 255, (batch, 2, 2, 16, 16), dtype=torch.uint8, device=dev)
    out = torch.full((batch * r * c + 64,), 7, dtype=torch.uint8, device=dev)
    hip.set_option("untilize_variant", 2)
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(out), batch, r, c, 1, hip.current_stream())
    assert torch.equal(out[:batch * r * c].view(batch, r, c), t[:, 0, 0, :r, :c]) and bool((out[batch * r * c:] == 7).all())


@pytest.mark.parametrize("fmt", [8, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_bfp_large_tensors(hip, dev, fmt, dtype):
    """Above the size up to which odd shapes go chunk by chunk (bf16 packs at any): what the generic kernel packs and unpacks."""
    hfmt, code = (hip.BFP8B if fmt == 8 else hip.BFP4B), (hip.F32 if dtype == torch.float32 else hip.BF16)
    shape = (1, 20500 if dtype == torch.float32 else 41000, 2051)
    assert shape[1] * shape[2] * dtype.itemsize > 160 << 20
    x = torch.randn(shape, device=dev, generator=torch.Generator(device=dev).manual_seed(4)).to(dtype)
    got = {}
    for variant in (0, 1):
        hip.set_option("pack_variant", variant)
        hip.set_option("unpack_variant", variant)
        try:
            p = pack_gpu(hip, dev, x, hfmt, shape, code, hip.ROW_MAJOR)
            got[variant] = p, unpack_gpu(hip, dev, p, hfmt, shape, code, hip.ROW_MAJOR)
        finally:
            hip.set_option("pack_variant", 0)
            hip.set_option("unpack_variant", 0)
    assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])


@pytest.mark.parametrize("fmt", [8, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_bfp_of_host_memory(hip, dev, fmt, dtype):
    """Either side in page-locked host memory, at a size from which that is packed and unpacked by strips: what the generic kernel makes of
    the same bits on the device, and nothing around it."""
    hfmt, code = (hip.BFP8B if fmt == 8 else hip.BFP4B), (hip.F32 if dtype == torch.float32 else hip.BF16)
    b, r, c = shape = (2, 1100, 2081)
    ints = torch.int32 if dtype == torch.float32 else torch.int16
    n, at, s = b * r * c, 3, hip.current_stream()
    bits = torch.randint(-2**15, 2**15 - 1, (n,), generator=torch.Generator().manual_seed(n)).to(ints)
    x = (bits << 16 if ints == torch.int32 else bits).to(dev)
    hip.set_option("pack_variant", 1)
    hip.set_option("unpack_variant", 1)
    try:
        packed = pack_gpu(hip, dev, x.view(dtype), hfmt, shape, code, hip.ROW_MAJOR)
        back = unpack_gpu(hip, dev, packed, hfmt, shape, code, hip.ROW_MAJOR).view(ints).reshape(-1)
        torch.cuda.synchronize()
    finally:
        hip.set_option("pack_variant", 0)
        hip.set_option("unpack_variant", 0)
    hx, hp = torch.full((n + 32,), 5, dtype=ints).pin_memory(), torch.full((packed.numel() + 32,), 9, dtype=torch.uint8).pin_memory()
    hx[at:at + n] = x.cpu()
    got = torch.zeros_like(packed)
    hip.call("ttm_bfp_pack", hip.ptr(hx[at:]), code, hip.ROW_MAJOR, hip.ptr(got), hfmt, b, r, c, s)
    hip.call("ttm_bfp_pack", hip.ptr(x), code, hip.ROW_MAJOR, hip.ptr(hp), hfmt, b, r, c, s)
    torch.cuda.synchronize()
    assert torch.equal(got, packed) and torch.equal(hp[:packed.numel()], packed.cpu()) and bool((hp[packed.numel():] == 9).all())
    dx = torch.full((n + 32,), 5, dtype=ints, device=dev)
    hip.call("ttm_bfp_unpack", hip.ptr(hp), hfmt, hip.ptr(dx[at:]), code, hip.ROW_MAJOR, b, r, c, s)
    hx.fill_(5)
    hip.call("ttm_bfp_unpack", hip.ptr(packed), hfmt, hip.ptr(hx[at:]), code, hip.ROW_MAJOR, b, r, c, s)
    torch.cuda.synchronize()
    for o in (dx.cpu(), hx):
        assert torch.equal(o[at:at + n], back.cpu()) and bool((o[:at] == 5).all()) and bool((o[at + n:] == 5).all())


def test_bfp_of_shapes_that_strips_could_serve_can_be_captured(hip, dev):
    """Which memory the pointers name is asked of such shapes, under capture as well."""
    b, r, c = shape = (2, 1100, 2081)
    x = torch.randn(b * r * c, device=dev)
    want = pack_gpu(hip, dev, x, hip.BFP8B, shape, hip.F32, hip.ROW_MAJOR)
    back = unpack_gpu(hip, dev, want, hip.BFP8B, shape, hip.F32, hip.ROW_MAJOR)
    p, y = torch.zeros_like(want), torch.zeros_like(back)
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        hip.call("ttm_bfp_pack", hip.ptr(x), hip.F32, hip.ROW_MAJOR, hip.ptr(p), hip.BFP8B, b, r, c, hip.current_stream())
        hip.call("ttm_bfp_unpack", hip.ptr(p), hip.BFP8B, hip.ptr(y), hip.F32, hip.ROW_MAJOR, b, r, c, hip.current_stream())
    for _ in range(3):
        p.zero_()
        y.zero_()
        g.replay()
        torch.cuda.synchronize()
        assert torch.equal(p, want) and torch.equal(y, back)


@pytest.mark.parametrize("rows,cols", [(41000, 2051), (41024, 2048)])
def test_large_tensors_take_strips(hip, dev, rows, cols):
    """Above the size up to which every shape goes chunk by chunk: whole strips and rows that start anywhere, against torch."""
    g = torch.Generator(device=dev).manual_seed(3)
    x = torch.randint(-2**15, 2**15 - 1, (rows, cols), dtype=torch.int16, device=dev, generator=g)
    pr, pc = -(-rows // 32) * 32, -(-cols // 32) * 32
    assert pr * pc * 2 > 160 << 20
    padded = torch.nn.functional.pad(x, (0, pc - cols, 0, pr - rows))
    want = padded.reshape(pr // 32, 2, 16, pc // 32, 2, 16).permute(0, 3, 1, 4, 2, 5).contiguous().reshape(-1)
    t = torch.full((pr * pc,), 0x55, dtype=torch.int16, device=dev)
    hip.call("ttm_tilize", hip.ptr(x), hip.ptr(t), 1, rows, cols, 2, hip.current_stream())
    assert torch.equal(t, want)
    back = torch.full((rows * cols + 64,), 7, dtype=torch.int16, device=dev)
    hip.call("ttm_untilize", hip.ptr(want), hip.ptr(back), 1, rows, cols, 2, hip.current_stream())
    assert torch.equal(back[:rows * cols].reshape(rows, cols), x) and bool((back[rows * cols:] == 7).all())


def test_c1_operands_layout(hip, dev, orc):
    a, b = datagen.c1_matmul()
    for m in (a, b):
        x = m.view(torch.int16).numpy().view(np.uint16)
        t = run_tilize(hip, dev, x)
        assert np.array_equal(t.cpu().numpy().view(np.uint16), orc.tilize(x))


def pack_gpu(hip, dev, xd, fmt, shape, dtype, layout):
    b, r, c = shape
    pr, pc = (r + 31) // 32 * 32, (c + 31) // 32 * 32
    nt = b * (pr // 32) * (pc // 32)
    out = torch.full((nt * hip.bfp_tile_bytes(fmt),), 0x55, dtype=torch.uint8, device=dev)
    hip.call("ttm_bfp_pack", hip.ptr(xd), dtype, layout, hip.ptr(out), fmt, b, r, c, hip.current_stream())
    return out


def unpack_gpu(hip, dev, pd, fmt, shape, dtype, layout):
    b, r, c = shape
    pr, pc = (r + 31) // 32 * 32, (c + 31) // 32 * 32
    n = b * r * c if layout == hip.ROW_MAJOR else b * pr * pc
    out = torch.full((n,), -7, dtype=torch.float32 if dtype == hip.F32 else torch.bfloat16, device=dev)
    hip.call("ttm_bfp_unpack", hip.ptr(pd), fmt, hip.ptr(out), dtype, layout, b, r, c, hip.current_stream())
    return out


@pytest.mark.parametrize("fmt", [8, 4])
@pytest.mark.parametrize("shape", [(1, 32, 32), (1, 256, 512), (2, 64, 96), (1, 40, 50), (3, 1, 33), (1, 1024, 1024)])
def test_bfp_pack_unpack_f32_rowmajor(hip, dev, orc, fmt, shape):
    hfmt = hip.BFP8B if fmt == 8 else hip.BFP4B
    x = datagen.c2_outliers(shape[0] * shape[1], shape[2], seed=3).reshape(shape)
    x[0, 0, : min(4, shape[2])] = 0.0
    xd = x.to(dev)
    pd = pack_gpu(hip, dev, xd, hfmt, shape, hip.F32, hip.ROW_MAJOR)
    want = orc.bfp_pack(x.numpy(), fmt)
    torch.cuda.synchronize()
    assert np.array_equal(pd.cpu().numpy(), want)
    back = unpack_gpu(hip, dev, pd, hfmt, shape, hip.F32, hip.ROW_MAJOR)
    torch.cuda.synchronize()
    want_back = orc.bfp_unpack(want, shape, fmt)
    assert np.array_equal(back.cpu().numpy().view(np.uint32), want_back.reshape(-1).view(np.uint32))


@pytest.mark.parametrize("fmt", [8, 4])
def test_bfp_tiled_and_bf16_sides(hip, dev, orc, fmt):
    hfmt = hip.BFP8B if fmt == 8 else hip.BFP4B
    shape = (2, 64, 128)
    x = datagen.c2_outliers(128, 128, seed=5).reshape(shape)
    xb = x.to(torch.bfloat16)
    want = orc.bfp_pack(xb.float().numpy(), fmt)          # bf16 sources are widened exactly
    # bf16 row-major source
    pd = pack_gpu(hip, dev, xb.to(dev), hfmt, shape, hip.BF16, hip.ROW_MAJOR)
    torch.cuda.synchronize()
    assert np.array_equal(pd.cpu().numpy(), want)
    # fp32 tile-ordered source
    tiled = torch.from_numpy(orc.tilize(xb.float().numpy())).to(dev)
    pd2 = pack_gpu(hip, dev, tiled, hfmt, shape, hip.F32, hip.TILE)
    # bf16 tile-ordered source
    pd3 = pack_gpu(hip, dev, tiled.to(torch.bfloat16), hfmt, shape, hip.BF16, hip.TILE)
    torch.cuda.synchronize()
    assert np.array_equal(pd2.cpu().numpy(), want) and np.array_equal(pd3.cpu().numpy(), want)
    # unpack to every plain side
    vals = orc.bfp_unpack(want, shape, fmt)
    u1 = unpack_gpu(hip, dev, pd, hfmt, shape, hip.BF16, hip.ROW_MAJOR)
    u2 = unpack_gpu(hip, dev, pd, hfmt, shape, hip.F32, hip.TILE)
    u3 = unpack_gpu(hip, dev, pd, hfmt, shape, hip.BF16, hip.TILE)
    torch.cuda.synchronize()
    assert np.array_equal(u1.float().cpu().numpy(), vals.reshape(-1))      # bf16 holds decoded values exactly
    assert np.array_equal(u2.cpu().numpy(), orc.tilize(vals))
    assert np.array_equal(u3.float().cpu().numpy(), orc.tilize(vals))


def test_bfp_special_values(hip, dev, orc):
    x = np.zeros((32, 32), dtype=np.float32)
    x[0, :8] = [1.0, 0.5, -0.25, 1.9921875, 1.984375, 0.0078125, -0.00390625, 0.01171875]
    x[1, :4] = [1e-40, -1e-39, 0.0, -0.0]                      # fp32 subnormals
    x[2, :3] = [3e38, -1e38, 1.0]
    x[3, :2] = [2.0 ** -120, 2.0 ** -126]
    x[4, :] = -0.0
    for fmt, hfmt in ((8, hip.BFP8B), (4, hip.BFP4B)):
        pd = pack_gpu(hip, dev, torch.from_numpy(x).to(dev), hfmt, (1, 32, 32), hip.F32, hip.ROW_MAJOR)
        torch.cuda.synchronize()
        want = orc.bfp_pack(x, fmt)
        assert np.array_equal(pd.cpu().numpy(), want)
        back = unpack_gpu(hip, dev, pd, hfmt, (1, 32, 32), hip.F32, hip.ROW_MAJOR)
        torch.cuda.synchronize()
        assert np.array_equal(back.cpu().numpy().view(np.uint32),
                              orc.bfp_unpack(want, (32, 32), fmt).reshape(-1).view(np.uint32))


def test_unpack_arbitrary_bytes(hip, dev, orc):
    """Every exponent/mantissa byte pattern decodes like the oracle (incl. 0x80 = -0 -> +0)."""
    rng = np.random.default_rng(9)
    for fmt, hfmt in ((8, hip.BFP8B), (4, hip.BFP4B)):
        tb = orc.bfp_tile_bytes(fmt)
        p = rng.integers(0, 256, size=16 * tb, dtype=np.uint8)
        p[:64] = np.arange(64) * 4            # low and high exponents, incl. 0 and 252
        p[tb: tb + 64] = 255 - np.arange(64)
        back = unpack_gpu(hip, dev, torch.from_numpy(p).to(dev), hfmt, (1, 128, 128), hip.F32, hip.TILE)
        torch.cuda.synchronize()
        want = orc.bfp_unpack_tiles(p, fmt)
        assert np.array_equal(back.cpu().numpy().view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("fmt", [8, 4])
def test_full_size_properties(hip, dev, orc, fmt):
    """Config 2 at 8192 x 8192: every packed tile and every unpacked value against the oracle, then round-trip properties."""
    hfmt = hip.BFP8B if fmt == 8 else hip.BFP4B
    W = 7 if fmt == 8 else 3
    x = datagen.c2_outliers(8192, 8192, seed=0)
    xd = x.to(dev)
    shape = (1, 8192, 8192)
    pd = pack_gpu(hip, dev, xd, hfmt, shape, hip.F32, hip.ROW_MAJOR)
    torch.cuda.synchronize()
    tb = hip.bfp_tile_bytes(hfmt)
    assert pd.numel() == 65536 * tb
    orc.set_threads(orc.max_threads())
    try:
        want_packed = orc.bfp_pack(x.numpy(), fmt)                 # all 65 536 tiles
        want_back = orc.bfp_unpack(want_packed, (8192, 8192), fmt)
    finally:
        orc.set_threads(1)
    assert np.array_equal(pd.cpu().numpy(), want_packed)
    y = unpack_gpu(hip, dev, pd, hfmt, shape, hip.F32, hip.ROW_MAJOR).reshape(8192, 8192)
    assert np.array_equal(y.cpu().numpy().view(np.uint32), want_back.view(np.uint32))
    del want_packed, want_back
    # idempotence: pack(unpack(pack(x))) == pack(x)
    pd2 = pack_gpu(hip, dev, y, hfmt, shape, hip.F32, hip.ROW_MAJOR)
    torch.cuda.synchronize()
    assert torch.equal(pd, pd2)
    # error bound per 16-element row: half a unit of the shared scale unless saturated
    xr, yr = xd.reshape(-1, 16), y.reshape(-1, 16)
    _, ex = torch.frexp(xr.abs().amax(dim=1))
    unit = torch.ldexp(torch.ones_like(ex, dtype=torch.float32), ex - 1 - (W - 1))[:, None]
    err = (xr - yr).abs()
    assert bool(torch.all(err <= unit))
    # (alignment bits are truncated before rounding, so a hair over half a unit is possible)
    assert bool(torch.all((err <= unit / 2 * (1 + 2.0 ** -16)) | (yr.abs() == unit * (2 ** W - 1))))
    # tilize -> untilize round trip and checksum preservation at full size
    t = torch.empty_like(xd)
    hip.call("ttm_tilize", hip.ptr(xd), hip.ptr(t), 1, 8192, 8192, 4, hip.current_stream())
    back = torch.empty_like(xd)
    hip.call("ttm_untilize", hip.ptr(t), hip.ptr(back), 1, 8192, 8192, 4, hip.current_stream())
    torch.cuda.synchronize()
    assert torch.equal(back, xd)
    assert int(t.view(torch.int32).to(torch.int64).sum()) == int(xd.view(torch.int32).to(torch.int64).sum())
    assert np.array_equal(t.reshape(-1).cpu().numpy(), orc.tilize(x.numpy()))


@pytest.mark.parametrize("fmt", [8, 4])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("shape,shift", [((1, 1, 1), 0), ((2, 33, 129), 1), ((1, 64, 255), 3), ((3, 31, 257), 0), ((1, 95, 1023), 5), ((2, 40, 300), 2),
                                         ((1, 32, 512), 1), ((1, 500, 384), 0), ((2, 1100, 2081), 7), ((2, 50, 83), 1), ((3, 70, 167), 5), ((2, 90, 16), 1), ((1, 70, 17), 3)])
def test_bfp_ragged(hip, dev, orc, fmt, dtype, shape, shift):
    """Rows that start and end anywhere, on buffers that start at any element: packed bytes and read-back of the rule's choice, the chunk
    kernel and the strips against the generic kernel, and of that against the oracle (random bit patterns: infinities, NaN and subnormal numbers among them), nothing written around them."""
    hfmt, code = (hip.BFP8B if fmt == 8 else hip.BFP4B), (hip.F32 if dtype == torch.float32 else hip.BF16)
    b, r, c = shape
    n, pad, s = b * r * c, 64, hip.current_stream()
    packed = b * ((r + 31) // 32) * ((c + 31) // 32) * hip.lib().ttm_bfp_tile_bytes(hfmt)
    ints = torch.int32 if dtype == torch.float32 else torch.int16
    limit = 2 ** (8 * ints.itemsize - 1)
    rng = np.random.default_rng(n)
    bits = torch.from_numpy(rng.integers(-limit, limit, n)).to(ints)
    plain = torch.randn(n, generator=torch.Generator().manual_seed(n)).to(dtype)
    for x, oracle in ((plain, True), (bits.view(dtype), False)):
        src = torch.zeros(n + 2 * pad, dtype=dtype, device=dev)
        src[pad + shift:pad + shift + n] = x.to(dev)
        got = {}
        for variant in (0, 1, 2, 3):
            hip.set_option("pack_variant", variant)
            hip.set_option("unpack_variant", variant)
            try:
                p = torch.full((packed + 32,), 9, dtype=torch.uint8, device=dev)
                hip.call("ttm_bfp_pack", hip.ptr(src[pad + shift:]), code, hip.ROW_MAJOR, hip.ptr(p), hfmt, b, r, c, s)
                back = torch.full((n + 2 * pad,), 5, dtype=ints, device=dev)
                hip.call("ttm_bfp_unpack", hip.ptr(p), hfmt, hip.ptr(back[pad + shift:]), code, hip.ROW_MAJOR, b, r, c, s)
                torch.cuda.synchronize()
            finally:
                hip.set_option("pack_variant", 0)
                hip.set_option("unpack_variant", 0)
            got[variant] = p.cpu(), back.cpu()
        p, back = got[1]
        for variant in (0, 2, 3):
            assert torch.equal(got[variant][0], p) and torch.equal(got[variant][1], back), variant
        assert (p[packed:] == 9).all() and (back[:pad + shift] == 5).all() and (back[pad + shift + n:] == 5).all()
        if oracle:
            want = orc.bfp_pack(x.float().numpy().reshape(shape), fmt)
            assert np.array_equal(p[:packed].numpy(), want)
            vals = orc.bfp_unpack(want, shape, fmt).reshape(-1)
            assert np.array_equal(back[pad + shift:pad + shift + n].view(dtype).float().numpy(), vals)


@pytest.mark.parametrize("shapes", [
    [(32, 4096, 2), (1, 128, 2), (1, 128, 2), (1, 16, 0), (1, 128, 0)],                       # a decode step's inputs
    [(33, 65, 4), (1, 1, 1), (31, 31, 2), (64, 1000, 1), (5, 7, 4), (200, 3, 2), (1, 1040, 0), (17, 129, 2)],
    [(0, 5, 2), (257, 9, 1)],
])
def test_tilize_group(hip, dev, shapes):
    """Several tensors in one launch against each by itself: every element size, ragged extents, copies, empty ones; from device and from
    page-locked memory, at odd element offsets too."""
    import ctypes

    class Item(ctypes.Structure):
        _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("rows", ctypes.c_int64), ("cols", ctypes.c_int64), ("elem", ctypes.c_int)]

    g = torch.Generator().manual_seed(len(shapes))
    for pinned in (False, True):
        items, want, got, keep = (Item * len(shapes))(), [], [], []
        for i, (rows, cols, elem) in enumerate(shapes):
            shift = 0 if elem == 0 else (i % 3) * elem      # rows that start at any element
            raw = torch.randint(0, 256, (shift + rows * cols * max(elem, 1) + 64,), generator=g, dtype=torch.uint8)
            raw = raw.pin_memory() if pinned else raw.to(dev)
            keep.append(raw)
            data = raw[shift:shift + rows * cols * max(elem, 1)].clone()
            n = rows * cols if elem == 0 else (rows + 31) // 32 * 32 * ((cols + 31) // 32 * 32) * elem
            out = torch.full((n,), 0xA5, dtype=torch.uint8, device=dev)
            if elem and n:
                ref, src = torch.full_like(out, 0x5A), data.to(dev)
                hip.call("ttm_tilize", hip.ptr(src), hip.ptr(ref), 1, rows, cols, elem, hip.current_stream())
            else:
                ref = data.to(dev)
            items[i] = Item(raw.data_ptr() + shift, out.data_ptr(), rows, cols, elem)
            want.append(ref)
            got.append(out)
        hip.call("ttm_tilize_group", items, len(shapes), hip.current_stream())
        torch.cuda.synchronize()
        for a, b in zip(got, want):
            assert torch.equal(a, b)


def test_tilize_group_refuses(hip, dev):
    import ctypes

    class Item(ctypes.Structure):
        _fields_ = [("src", ctypes.c_void_p), ("dst", ctypes.c_void_p), ("rows", ctypes.c_int64), ("cols", ctypes.c_int64), ("elem", ctypes.c_int)]

    t = torch.zeros(4096, dtype=torch.uint8, device=dev)
    p = t.data_ptr()
    for bad in (Item(p, p, 1, 8, 3), Item(p, p + 8, 1, 8, 2), Item(p + 1, p, 1, 8, 2), Item(p, p, 1, 24, 0), Item(None, p, 1, 16, 0), Item(p, p, -1, 8, 2), Item(p, p, 2, 16, 0)):
        with pytest.raises(hip.TTMError):
            hip.call("ttm_tilize_group", (Item * 1)(bad), 1, hip.current_stream())
    with pytest.raises(hip.TTMError):
        hip.call("ttm_tilize_group", (Item * 9)(), 9, hip.current_stream())
