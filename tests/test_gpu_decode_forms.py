"""The two forms of the decode attention kernel (one workgroup per user and kv head; equal shares of all users' visible tiles) at the
edges of both: users with no visible key, contexts that end inside a tile, more shares than tiles, more than 64 users, windows,
pages, sinks, head dims with and without a kernel of their own.  Each form against the oracle within a bf16 step of outputs below
1 (2^-7) plus the bf16 rounding of the softmax numerators (2^-8 of the largest value row, |v| < 5: 2^-6 together)."""
import numpy as np
import pytest
import torch

from ttmlir_amd import datagen
from test_gpu_linear import tilize_dev, untilize_dev

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("form", [1, 2])
@pytest.mark.parametrize("B,H,Hkv,S,D,cur,window,sink", [
    (1, 4, 1, 32, 128, [0], -1, False),                        # one key
    (3, 8, 2, 512, 64, [511, 31, 32], -1, False),
    (2, 16, 2, 256, 128, [7, 255], 33, True),                  # eight heads per kv head
    (70, 4, 2, 96, 32, [(17 * u) % 96 for u in range(70)], -1, False),
    (2, 3, 1, 160, 96, [159, 3], -1, True),                    # no kernel of its own
    (2, 2, 2, 1024, 256, [1000, 64], -1, False),
    (2, 4, 4, 64, 128, [-1, 40], -1, False),                   # a user that sees nothing
    (2, 4, 1, 4096, 128, [4095, 2000], -1, True),              # more pieces of a user than are requested ahead of their weights
    (2, 8, 1, 8192, 256, [8191, 8000], -1, False),             # ... with a lane per column
    (2, 4, 1, 4096, 64, [100, 40], -1, False),                 # most shares empty
    (1, 2, 1, 65536, 32, [65535], -1, False),                  # as many pieces as there are shares
])
def test_both_forms_against_the_oracle(hip, dev, orc, form, B, H, Hkv, S, D, cur, window, sink):
    q, k, v = (datagen.randn(s, seed=i, dtype=torch.bfloat16) for i, s in enumerate(((1, B, H, D), (B, Hkv, S, D), (B, Hkv, S, D))))
    sk = datagen.randn((H, 1), seed=9, dtype=torch.bfloat16) if sink else None
    qt, kt, vt = (tilize_dev(hip, t, dev) for t in (q, k, v))
    st = tilize_dev(hip, sk, dev) if sink else None
    cp = torch.tensor(cur, dtype=torch.int32, device=dev)
    out = torch.full_like(qt, float("nan"))
    hip.set_option("sdpa_decode_form", form)
    try:
        hip.call("ttm_sdpa_decode_windowed", hip.ptr(qt), hip.ptr(kt), hip.ptr(vt), hip.ptr(cp), None, 1, 1, None, 0, 0, 0, hip.ptr(out),
                 hip.BF16, B, H, Hkv, S, D, 1, 0.0, 0, window, hip.ptr(st) if sink else None, hip.current_stream())
        torch.cuda.synchronize()
    finally:
        hip.set_option("sdpa_decode_form", 0)
    got = untilize_dev(hip, out, (1, B, H, D), dev).float().cpu().numpy()
    seen = [i for i, c in enumerate(cur) if c >= 0]
    want = orc.sdpa_decode(q.float().numpy()[:, seen], k.float().numpy()[seen], v.float().numpy()[seen], cur_pos=[cur[i] for i in seen],
                           is_causal=True, sliding_window=window if window >= 0 else None,
                           attention_sink=sk.float().numpy() if sink else None)
    assert np.max(np.abs(got[:, seen] - want)) <= 2.0 ** -6
    assert not got[:, [i for i, c in enumerate(cur) if c < 0]].any()
