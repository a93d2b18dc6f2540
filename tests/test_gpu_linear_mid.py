"""The mid-size linear kernel under every plan it can take (row tiles and K shares per workgroup, slices of K), at the edges of its
tiles: ragged rows, columns and K, fewer k-tiles than shares, one column tile, more rows than a workgroup holds; groups and the
gated form against separate launches of the same plan.  Against the CPU oracle on the weights the device multiplies; outputs are
O(1), so one bf16 step is at most 2^-6 and the accumulation order adds less than that (2^-5 as in the other linear tests)."""
import ctypes

import numpy as np
import pytest
import torch

from ttmlir_amd import datagen
from test_gpu_linear import check, metrics, pack_weight, run_linear, tilize_dev, untilize_dev  # noqa: F401 (metrics: fixture)

pytestmark = pytest.mark.gpu
PLANS = [8101, 8102, 8201, 8202, 4201, 4204, 8401, 8404]


@pytest.fixture
def plan(hip, request):
    hip.set_option("linear_mid", request.param)
    yield request.param
    hip.set_option("linear_mid", 0)


@pytest.mark.parametrize("plan", PLANS, indirect=True)
@pytest.mark.parametrize("wfmt_name", ["bfp8", "bfp4", "bf16", "bf16_nk"])
@pytest.mark.parametrize("M,K,N,act,bias", [(33, 37 * 32 + 11, 5 * 32 + 7, "silu", True), (161, 70, 32, None, False), (1, 1030, 100, "gelu", True)])
def test_every_plan_against_the_oracle(hip, dev, orc, metrics, plan, wfmt_name, M, K, N, act, bias):  # noqa: F811
    wfmt = {"bfp8": hip.BFP8B, "bfp4": hip.BFP4B}.get(wfmt_name, hip.BF16)
    a = datagen.randn((M, K), seed=M, dtype=torch.bfloat16)
    w = datagen.randn((K, N), seed=N, std=K ** -0.5)
    b = datagen.randn((N,), seed=7, std=0.5, dtype=torch.bfloat16) if bias else None
    nk = wfmt_name == "bf16_nk"
    got, w_eff = run_linear(hip, dev, a, w.t().contiguous() if nk else w, b, act, wfmt, transpose_w=nk)
    check(orc, metrics, got, a, w_eff, b, act, max_abs=2.0 ** -5)


@pytest.mark.parametrize("plan", [8101, 8202, 4201, 8404], indirect=True)
def test_batches_and_groups_equal_separate_launches(hip, dev, plan):
    M, K, Ns = 70, 300, (200, 40, 96)
    a = datagen.randn((M, K), seed=1, dtype=torch.bfloat16)
    ws = [datagen.randn((K, N), seed=2 + i, std=0.05) for i, N in enumerate(Ns)]
    want = [run_linear(hip, dev, a, w, None, None, hip.BFP8B)[0] for w in ws]
    at, wt = tilize_dev(hip, a, dev), [pack_weight(hip, w, hip.BFP8B, dev) for w in ws]
    outs = [torch.full((96 * ((N + 31) // 32 * 32),), float("nan"), dtype=torch.bfloat16, device=dev) for N in Ns]
    arr = lambda t, v: (t * len(v))(*v)
    hip.call("ttm_linear_group", hip.ptr(at), 3, arr(ctypes.c_void_p, [t.data_ptr() for t in wt]), hip.BFP8B,
             arr(ctypes.c_void_p, [t.data_ptr() for t in outs]), arr(ctypes.c_int64, Ns), None, M, K, hip.current_stream())
    for o, N, w in zip(outs, Ns, want):
        assert torch.equal(untilize_dev(hip, o, (M, N), dev).cpu(), w)
    three, _ = run_linear(hip, dev, a.expand(3, M, K), datagen.randn((3, K, 64), seed=9, std=0.05), None, None, hip.BFP4B)
    for i in range(3):
        one, _ = run_linear(hip, dev, a, datagen.randn((3, K, 64), seed=9, std=0.05)[i], None, None, hip.BFP4B)
        assert torch.equal(three[i], one)


@pytest.mark.parametrize("plan", [4201, 4401], indirect=True)
@pytest.mark.parametrize("M,K,N", [(65, 64, 104), (65, 512, 5760)])
def test_gated_form_against_the_oracle(hip, dev, orc, plan, M, K, N):
    a = datagen.randn((M, K), seed=1, dtype=torch.bfloat16)
    ws = [datagen.randn((K, N), seed=2 + i, std=K ** -0.5) for i in range(2)]
    at, wt = tilize_dev(hip, a, dev), [pack_weight(hip, w, hip.BFP8B, dev) for w in ws]
    out = torch.full(((M + 31) // 32 * 32 * ((N + 31) // 32 * 32),), float("nan"), dtype=torch.bfloat16, device=dev)
    assert hip.lib().ttm_linear_glu_supported(hip.BFP8B, M, N, K) == 1
    hip.call("ttm_linear_glu", hip.ptr(at), hip.ptr(wt[0]), hip.ptr(wt[1]), hip.BFP8B, hip.ptr(out), M, N, K, hip.ACT["silu"], 0, hip.current_stream())
    got = untilize_dev(hip, out, (M, N), dev).float().cpu().numpy()
    q = lambda w: orc.bfp_unpack(orc.bfp_pack(w.numpy(), 8), w.shape, 8)
    r, an = orc.round_bf16, a.float().numpy()
    ref = r(r(orc.linear(an, q(ws[0]), None, "silu")) * r(orc.linear(an, q(ws[1]))))
    # two factors of up to 4, each within a bf16 step (2^-6 at magnitudes below 4) of the oracle's, and the product's own step
    assert np.max(np.abs(got - ref)) <= 2.0 ** -3
    assert np.mean(got == ref) >= 0.97


@pytest.mark.parametrize("plan", [8101, 8201, 8401, 4201], indirect=True)
@pytest.mark.parametrize("wfmt_name", ["bfp8", "bfp4", "bf16"])
def test_infinite_activations(hip, dev, plan, wfmt_name):
    """An infinite activation gives the infinities and NaN (0 x inf) of its products with the weights the device holds."""
    M, K, N = 97, 160, 96
    a = datagen.randn((M, K), seed=3, dtype=torch.bfloat16)
    a[5, 40] = float("inf")
    a[70, 159] = float("-inf")
    w = datagen.randn((K, N), seed=4, std=0.1)
    got, w_eff = run_linear(hip, dev, a, w, None, None, {"bfp8": hip.BFP8B, "bfp4": hip.BFP4B}.get(wfmt_name, hip.BF16))
    want = a.float() @ torch.as_tensor(w_eff).float()
    got = got.float()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    assert torch.equal(torch.isinf(got), torch.isinf(want)) and torch.equal(got[torch.isinf(got)], want[torch.isinf(want)])


@pytest.mark.parametrize("plan", [8102, 8216, 8404], indirect=True)
@pytest.mark.parametrize("K", [20, 70])
def test_more_slices_than_k_tiles(hip, dev, orc, metrics, plan, K):  # noqa: F811
    a, w = datagen.randn((70, K), seed=1, dtype=torch.bfloat16), datagen.randn((K, 96), seed=2, std=K ** -0.5)
    got, w_eff = run_linear(hip, dev, a, w, None, None, hip.BFP8B)
    check(orc, metrics, got, a, w_eff, None, None, max_abs=2.0 ** -5)


@pytest.mark.parametrize("wfmt_name,M,K,N", [("bf16", 20, 4096, 512), ("bf16", 1, 2048, 128), ("bfp8", 100, 4096, 256)])
def test_a_split_product_is_recorded_on_a_stream_without_workspace(hip, dev, orc, metrics, wfmt_name, M, K, N):  # noqa: F811
    """Recorded as the first call of its stream and replayed on changing activations, with eager calls in between."""
    wfmt = {"bfp8": hip.BFP8B, "bf16": hip.BF16}[wfmt_name]
    w = datagen.randn((K, N), seed=N, std=K ** -0.5)
    xs = [datagen.randn((M, K), seed=i, dtype=torch.bfloat16) for i in range(3)]
    eager, w_eff = zip(*[run_linear(hip, dev, x, w, None, None, wfmt) for x in xs])
    wt = tilize_dev(hip, w.to(torch.bfloat16), dev) if wfmt == hip.BF16 else pack_weight(hip, w, wfmt, dev)
    a, out = tilize_dev(hip, xs[0], dev), torch.full(((M + 31) // 32 * 32 * N,), float("nan"), dtype=torch.bfloat16, device=dev)
    torch.cuda.synchronize()
    stream, graph, nodes = ctypes.c_void_p(), ctypes.c_void_p(), ctypes.c_size_t()
    hip.call("ttm_stream_create", ctypes.byref(stream))
    hip.call("ttm_graph_begin_capture", stream)
    try:
        hip.call("ttm_linear", hip.ptr(a), hip.BF16, hip.ptr(wt), wfmt, 0, None, hip.BF16, hip.TILE, hip.ptr(out), hip.BF16, 1, 1, M, N, K, 0, stream)
    finally:
        hip.call("ttm_graph_end_capture", stream, ctypes.byref(graph), ctypes.byref(nodes))
    assert nodes.value == 1
    for x, e in zip(xs, eager):
        a.copy_(tilize_dev(hip, x, dev))
        torch.cuda.synchronize()
        hip.call("ttm_graph_launch", graph, stream)
        hip.call("ttm_stream_sync", stream)
        got = untilize_dev(hip, out, (M, N), dev).cpu()
        check(orc, metrics, got, x, w_eff[0], None, None, max_abs=2.0 ** -5)
        assert torch.allclose(got.float(), e.float(), atol=2.0 ** -5)
    hip.call("ttm_graph_destroy", graph)
    hip.call("ttm_stream_destroy", stream)


@pytest.mark.parametrize("wfmt_name", ["bfp8", "bfp4"])
@pytest.mark.parametrize("M", [33, 64])
def test_infinite_activations_up_to_64_rows(hip, dev, wfmt_name, M):
    """The two-term operand leaves inf - inf in every column of such a row, here as in the decode kernel (which these sizes went to
    before); other rows are those of a call without it."""
    a = datagen.randn((M, 512), seed=3, dtype=torch.bfloat16)
    w, wfmt = datagen.randn((512, 96), seed=4, std=0.1), {"bfp8": hip.BFP8B, "bfp4": hip.BFP4B}[wfmt_name]
    clean, _ = run_linear(hip, dev, a, w, None, None, wfmt)
    a[5, 40], a[M - 1, 511] = float("inf"), float("-inf")
    hit = torch.zeros(M, dtype=torch.bool)
    hit[[5, M - 1]] = True
    for option in (0, 8101, 1):
        hip.set_option("linear_mid", option)
        try:
            got, _ = run_linear(hip, dev, a, w, None, None, wfmt)
        finally:
            hip.set_option("linear_mid", 0)
        assert torch.isnan(got[hit]).all() and torch.isfinite(got[~hit]).all()
        if option == 0:
            assert torch.equal(got[~hit], clean[~hit])


def _bfp4_weights(tiles):
    """float64 values of bfp4_b tiles [K / 32, N / 32, 576]."""
    kt, nt = tiles.shape[:2]
    face = tiles[:, :, 64:].reshape(kt, nt, 2, 2, 16, 8)
    nibbles = torch.stack([face & 15, face >> 4], -1).reshape(kt, nt, 2, 2, 16, 16).double()
    value = torch.where(nibbles >= 8, 8 - nibbles, nibbles) * 2.0 ** (tiles[:, :, :64].reshape(kt, nt, 2, 2, 16, 1).double() - 129)
    return value.permute(0, 2, 4, 1, 3, 5).reshape(kt * 32, nt * 32)


def _bfp4_product(hip, dev, a, tiles, options):
    M, K, N = a.shape[0], a.shape[1], tiles.shape[1] * 32
    at, wd = tilize_dev(hip, a, dev), tiles.reshape(-1).to(dev)
    out = torch.full(((M + 31) // 32 * 32 * N,), float("nan"), dtype=torch.bfloat16, device=dev)
    for name, v in options.items():
        hip.set_option(name, v)
    try:
        hip.call("ttm_linear", hip.ptr(at), hip.BF16, hip.ptr(wd), hip.BFP4B, 0, None, hip.BF16, hip.TILE, hip.ptr(out), hip.BF16, 1, 1, M, N, K, 0,
                 hip.current_stream())
    finally:
        for name in options:
            hip.set_option(name, 0)
    return untilize_dev(hip, out, (M, N), dev).cpu().double()


# the kernels that keep weights in registers, the decode kernel and the mid-size one under every kind of plan; the fused kernel, whose last step of two
# k-tiles reaches past an odd number of them, whole and in slices of K; and weights as images first
BFP4_FORMS = [(1, {}), (32, {}), (32, {"linear_decode_wide": 2}), (32, {"linear_decode_split": 3}), (64, {"linear_mid": 8101}), (100, {"linear_mid": 4201}),
              (130, {"linear_mid": 8202}), (128, {"linear_mid": 8401}), (352, {"linear_mid": 1, "linear_two_pass": 1}),
              (352, {"linear_mid": 1, "linear_two_pass": 1, "linear_split_k": 2}), (352, {"linear_mid": 1, "linear_two_pass": 2})]


@pytest.mark.parametrize("M,options", BFP4_FORMS)
def test_bfp4_operands_of_every_exponent(hip, dev, M, options):
    """Every nibble under every exponent as these kernels turn it into bf16: rows of the identity times such weights give them back, exactly from
    exponent 3 on and below at most 2^-127 too small, or as zeros by way of images.  (Those take 254 for an overflow.)"""
    K, N = 352, 96
    images = options.get("linear_two_pass") == 2
    g = torch.Generator().manual_seed(M)
    tiles = torch.randint(0, 256, (K // 32, N // 32, 576), generator=g, dtype=torch.uint8)
    tiles[:, :, :64] = (torch.arange(K // 32 * N // 32 * 64) % (254 if images else 255)).reshape(K // 32, N // 32, 64).to(torch.uint8)
    w = _bfp4_weights(tiles)
    small = tiles.clone()
    small[:, :, 64:] = torch.where(tiles[:, :, :64].repeat_interleave(8, -1) < 3, tiles[:, :, 64:], 0)
    small = _bfp4_weights(small)      # the weights below exponent 3, zeros elsewhere
    for rows in torch.randperm(K, generator=g).split(M)[:12]:
        a = torch.zeros(M, K, dtype=torch.bfloat16)
        a[torch.arange(len(rows)), rows] = 1.0
        got, want, below = _bfp4_product(hip, dev, a, tiles, options)[:len(rows)], w[rows], small[rows]
        assert torch.equal(got[below == 0], want[below == 0])
        if images:
            assert not got[below != 0].any()
        off = (want - got)[below != 0] * below[below != 0].sign()
        assert (off >= 0).all() and (images or (off <= 2.0 ** -127).all())


@pytest.mark.parametrize("options", [{}, {"linear_split_k": 2}])
def test_bfp4_fused_ends_with_its_k_tiles(hip, dev, options):
    """The last step of the fused kernel multiplies two k-tiles; where their number is odd the second is the last one again, under weights of
    zero: with the smallest exponents and activations of 2^100 nothing of it shows."""
    M, K, N = 352, 352, 96
    tiles = torch.randint(0, 256, (K // 32, N // 32, 576), generator=torch.Generator().manual_seed(7), dtype=torch.uint8)
    tiles[:, :, :64] = 3
    a = torch.zeros(M, K, dtype=torch.bfloat16)
    a[torch.arange(M), torch.arange(M)] = 2.0 ** 100
    got = _bfp4_product(hip, dev, a, tiles, {"linear_mid": 1, "linear_two_pass": 1, **options})
    assert torch.equal(got, _bfp4_weights(tiles) * 2.0 ** 100)


@pytest.mark.parametrize("M,options", BFP4_FORMS[:-1])
def test_bfp4_rows_of_exponent_255(hip, dev, M, options):
    """A row of weights that had an infinity or a NaN, under activations of 1: magnitude 4 is an infinity again, 5 to 7 are NaN, the others values like
    any."""
    K, N, k = 352, 96, 331
    tiles = torch.zeros(K // 32, N // 32, 576, dtype=torch.uint8)
    tiles[:, :, :64] = 120
    r = k % 32
    for half in (0, 1):
        f = (r >> 4) * 2 + half
        tiles[k // 32, :, f * 16 + (r & 15)] = 255
        tiles[k // 32, :, 64 + f * 128 + (r & 15) * 8:][:, :8] = torch.tensor([0x10 + 0x22 * j for j in range(8)], dtype=torch.uint8)   # 0 .. 15
    want = _bfp4_weights(tiles)[k]
    mag = want.abs() / 2.0 ** 126
    want[mag == 4] *= float("inf")
    want[mag > 4] = float("nan")
    assert want.isinf().sum() == 12 and want.isnan().sum() == 36
    got = _bfp4_product(hip, dev, torch.ones(M, K, dtype=torch.bfloat16), tiles, options)
    assert torch.equal(got.nan_to_num(1.0, 2.0 ** 200, -2.0 ** 200), want.nan_to_num(1.0, 2.0 ** 200, -2.0 ** 200).expand(M, N))
