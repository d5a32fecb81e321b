"""More key splits than the merge holds in registers at once (8): late chunks of a 4096-position context, over
both cache types, with splits that some rows do not see."""

import numpy as np
import pytest

from conftest import assert_close
from oracle.decode import prefill_attention
from test_gpu_prefill_attention import D, THETA, PrefillDims, run

pytestmark = pytest.mark.gpu

CTX = 4096


@pytest.mark.parametrize("cache", ["f32", "f16"])
# 16 splits, 15, 15 (f16 11), 10 (f16 8), 8, 10
@pytest.mark.parametrize("begin,n,heads,kv_heads", [(4095, 1, 14, 2), (3800, 17, 14, 2), (3700, 130, 8, 8),
                                                     (3800, 256, 14, 2), (3000, 1096, 4, 2), (2600, 70, 12, 12)])
def test_many_splits(device, begin, n, heads, kv_heads, cache):
    rng = np.random.default_rng(5 + begin + n)
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)
    q, k, v = f(n, heads * D), f(n, kv_heads * D), f(n, kv_heads * D)
    kc, vc = f(CTX, kv_heads, D), f(CTX, kv_heads, D)
    if cache == "f16":
        kc, vc = (c.astype(np.float16).astype(np.float32) for c in (kc, vc))
    given = [c.copy() if cache == "f32" else c.astype(np.float16).view(np.uint16) for c in (kc, vc)]
    dims = PrefillDims(n, begin + n, begin, heads, kv_heads, D, CTX, THETA)
    got = run(device, q, k, v, *given, begin, dims=dims)[1]
    want = prefill_attention(q, k, v, kc, vc, begin, heads, kv_heads, D, THETA, cache=cache)[1]
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    # f32 sums; f16: q and the softmax weights are rounded (2^-11 each)
    bar = (1e-5 * rms, 2e-5) if cache == "f32" else (1e-2 * rms, 1e-2)
    assert_close(got.ravel(), want.ravel(), *bar, label=f"{cache} begin {begin} n {n} heads {heads}/{kv_heads}")
