"""Which form causal attention over as many keys as queries takes (four or eight wavefronts per workgroup), on both sides of its lines: the
result is that form's bit for bit, and both lie within a bf16 step of outputs below 4 (2^-6) plus the bf16 rounding of the
probabilities (2^-8 of the largest value, below 6: 2^-5 together) of attention in float32."""
import pytest
import torch

from ttmlir_amd import datagen
from test_gpu_linear import tilize_dev, untilize_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("B,H,Hkv,S,D,window,four", [
    (1, 8, 8, 66, 128, -1, True),        # one block per matrix
    (1, 8, 4, 200, 128, -1, True),       # two, 128 columns
    (1, 8, 4, 200, 64, -1, False),       # and 64
    (1, 8, 8, 300, 64, -1, False),       # three blocks on a device that is not full
    (4, 32, 8, 300, 64, -1, True),       # 1.5 blocks per CU
    (2, 32, 8, 1100, 64, -1, True),      # 2.25, columns of nine
    (1, 32, 32, 1700, 128, -1, False),   # 1.75, columns of 14
    (4, 32, 8, 616, 128, -1, True),      # 2.5, columns of five
    (1, 32, 8, 1100, 64, 130, True),     # a window, more blocks than CUs
    (1, 32, 8, 500, 128, 60, False),     # a window, fewer
    (1, 16, 4, 8200, 128, -1, False),    # more than 4096 tokens, too few matrices for nine half rounds of blocks
    (1, 32, 32, 5125, 64, -1, False),    # enough of them, five blocks per CU
    (1, 32, 8, 7000, 64, -1, False),     # just under seven
    (2, 32, 8, 4200, 64, -1, True),      # 8.25
    (1, 16, 4, 4120, 128, 1024, False),  # a window, two rounds
    (2, 16, 4, 4120, 64, 500, True),     # a window, four
])
def test_form_by_the_rule(hip, dev, B, H, Hkv, S, D, window, four):
    q, k, v = (datagen.randn((B, n, S, D), seed=i, dtype=torch.bfloat16) for i, n in enumerate((H, Hkv, Hkv)))
    qt, kt, vt = (tilize_dev(hip, t, dev) for t in (q, k, v))
    got = {}
    for variant in (0, 7, 8):
        out = torch.full_like(qt, float("nan"))
        hip.set_option("sdpa_variant", variant)
        try:
            hip.call("ttm_sdpa_windowed", hip.ptr(qt), hip.ptr(kt), hip.ptr(vt), None, 1, 1, hip.ptr(out), hip.BF16, B, H, Hkv, S, S, D, 1, 0.0, 0,
                     window, None, hip.current_stream())
            torch.cuda.synchronize()
        finally:
            hip.set_option("sdpa_variant", 0)
        got[variant] = untilize_dev(hip, out, (B, H, S, D), dev).float()
    assert torch.equal(got[0], got[7 if four else 8])
    ref = lambda t: t.to(dev).float().repeat_interleave(H // t.shape[1], 1)
    i, j = torch.arange(S, device=dev)[:, None], torch.arange(S, device=dev)[None]
    hidden = (j > i) | ((j <= i - window) if window >= 0 else False)
    for b in range(B):
        scores = (ref(q[b:b + 1]) @ ref(k[b:b + 1]).transpose(-1, -2).contiguous() / D ** 0.5).masked_fill(hidden, float("-inf"))
        want = torch.softmax(scores, -1) @ ref(v[b:b + 1])
        for g in got.values():
            assert (g[b] - want[0]).abs().max() <= 2.0 ** -5
