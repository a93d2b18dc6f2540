"""Single query blocks against pairs of them in causal attention: the same numbers bit for bit, for odd and even counts of blocks,
numbers of (batch entry, kv head) that are and are not a multiple of the XCDs, windows, a sink, and more blocks than CUs; and both
against attention in float32 within a bf16 step of outputs below 4 (2^-6) plus the bf16 rounding of the probabilities (2^-8 of
the largest value, below 6: 2^-5 together)."""
import pytest
import torch

from ttmlir_amd import datagen
from test_gpu_linear import tilize_dev, untilize_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,S,D,window,sink", [
    (1, 8, 8, 129, 128, -1, False),      # two blocks, the second of one query
    (1, 4, 2, 640, 64, -1, True),        # five blocks, two kv heads
    (3, 6, 3, 300, 128, 100, False),     # nine groups, a window
    (2, 16, 4, 513, 64, -1, False),      # eight groups
    (1, 4, 4, 257, 32, -1, False),       # a head dim without the pipelined kernel
    (1, 48, 8, 800, 64, -1, False),      # 336 blocks
    (1, 32, 8, 1100, 128, 150, True),    # 288 blocks
])
def test_single_blocks_equal_pairs(hip, dev, B, H, Hkv, S, D, window, sink):
    q, k, v = (datagen.randn((B, n, S, D), seed=i, dtype=torch.bfloat16) for i, n in enumerate((H, Hkv, Hkv)))
    sk = datagen.randn((1, H, 1, 1), seed=9, dtype=torch.bfloat16) if sink else None
    qt, kt, vt = (tilize_dev(hip, t, dev) for t in (q, k, v))
    st = tilize_dev(hip, sk, dev) if sink else None
    got = []
    for variant in (9, 10, 0):
        out = torch.full_like(qt, float("nan"))
        hip.set_option("sdpa_variant", variant)
        try:
            hip.call("ttm_sdpa_windowed", hip.ptr(qt), hip.ptr(kt), hip.ptr(vt), None, 1, 1, hip.ptr(out), hip.BF16, B, H, Hkv, S, S, D, 1, 0.0, 0,
                     window, hip.ptr(st) if sink else None, hip.current_stream())
            torch.cuda.synchronize()
        finally:
            hip.set_option("sdpa_variant", 0)
        got.append(untilize_dev(hip, out, (B, H, S, D), dev).float().cpu())
    assert torch.equal(got[0], got[1])
    ref = lambda t: t.float().repeat_interleave(H // t.shape[1], 1)
    scores = ref(q) @ ref(k).transpose(-1, -2) / D ** 0.5
    i, j = torch.arange(S)[:, None], torch.arange(S)[None]
    scores = scores.masked_fill((j > i) | ((j <= i - window) if window >= 0 else False), float("-inf"))
    if sink:
        scores = torch.cat([scores, (sk.float() / D ** 0.5).expand(B, H, S, 1)], -1)
    want = torch.softmax(scores, -1)[..., :S] @ ref(v)
    for g in got[1:]:
        assert (g - want).abs().max() <= 2.0 ** -5
