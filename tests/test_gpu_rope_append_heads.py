"""The chunk attention's RoPE and cache append where a thread's pairs read ahead of the angles are fewer
than, exactly and more than the row's (16 heads of q and k are all of them)."""

import numpy as np
import pytest

from oracle.decode import prefill_attention
from test_gpu_prefill_attention import CTX, D, THETA, run

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cache", ["f32", "f16"])
@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (8, 8), (15, 3), (24, 8)])
def test_rows_rotated_and_appended(device, heads, kv_heads, cache):
    rng = np.random.default_rng(9 + heads)
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)
    n, begin = 5, 1001
    q, k, v = f(n, heads * D), f(n, kv_heads * D), f(n, kv_heads * D)
    kc, vc = (f(CTX, kv_heads, D).astype(np.float16).astype(np.float32) for _ in range(2))
    given = [c.copy() if cache == "f32" else c.astype(np.float16).view(np.uint16) for c in (kc, vc)]
    got_q, _, got_k, got_v = run(device, q, k, v, *given, begin, heads=heads, kv_heads=kv_heads)
    want_q, _ = prefill_attention(q, k, v, kc, vc, begin, heads, kv_heads, D, THETA, cache=cache)  # appends to kc, vc
    # the double-precision angle may differ in its last bit between GPU and host: one ulp of the f32 result
    np.testing.assert_array_max_ulp(got_q, want_q, maxulp=1)
    if cache == "f32":
        np.testing.assert_array_max_ulp(got_k, kc, maxulp=1)
        np.testing.assert_array_equal(got_v, vc)
    else:
        got_k, got_v = (a.view(np.float16).astype(np.float32) for a in (got_k, got_v))
        np.testing.assert_array_max_ulp(got_k.astype(np.float16), kc.astype(np.float16), maxulp=1)
        np.testing.assert_array_equal(got_v, vc.astype(np.float16).astype(np.float32))
