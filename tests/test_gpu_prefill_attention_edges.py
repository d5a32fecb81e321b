"""The chunk attention at the edges of its tiles (64 queries, 64 keys, key splits), over both cache types, and
values that must not reach the queries that do not see them."""

import numpy as np
import pytest

from conftest import assert_close
from oracle.decode import prefill_attention
from test_gpu_prefill_attention import CTX, D, THETA, run

pytestmark = pytest.mark.gpu


def inputs(n, heads, kv_heads, seed):
    rng = np.random.default_rng(seed)
    f = lambda *s: rng.standard_normal(s, dtype=np.float32)
    return f(n, heads * D), f(n, kv_heads * D), f(n, kv_heads * D), f(CTX, kv_heads, D), f(CTX, kv_heads, D)


# one query at the first, the last and a tile's first key; 64 and 65 queries; chunks whose keys split
# (5, 7 and 8 splits, some empty for some rows), one head per kv head. The f16 bar is the one of the
# f16 kernel's own test: q and the softmax weights are rounded to f16 (2^-11 each).
@pytest.mark.parametrize("cache", ["f32", "f16"])
@pytest.mark.parametrize("begin,n,heads,kv_heads", [(0, 1, 14, 2), (64, 1, 14, 2), (2047, 1, 14, 2), (0, 65, 2, 2),
                                                     (63, 64, 3, 3), (1792, 256, 14, 2), (1000, 17, 8, 1), (0, 600, 4, 4)])
def test_tile_edges(device, begin, n, heads, kv_heads, cache):
    q, k, v, kc, vc = inputs(n, heads, kv_heads, 31 + begin + n)
    if cache == "f16":
        kc, vc = (c.astype(np.float16).astype(np.float32) for c in (kc, vc))
    given = [c.copy() if cache == "f32" else c.astype(np.float16).view(np.uint16) for c in (kc, vc)]
    got = run(device, q, k, v, *given, begin, heads=heads, kv_heads=kv_heads)[1]
    want = prefill_attention(q, k, v, kc, vc, begin, heads, kv_heads, D, THETA, cache=cache)[1]
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    bar = (1e-5 * rms, 2e-5) if cache == "f32" else (1e-2 * rms, 1e-2)
    assert_close(got.ravel(), want.ravel(), *bar, label=f"{cache} begin {begin} n {n} heads {heads}/{kv_heads}")


@pytest.mark.parametrize("begin,n,bad", [(0, 100, 70), (1800, 100, 33)])
def test_later_rows_of_infinity_and_nan_stay_unseen(device, begin, n, bad):
    """Row `bad` of the chunk holds NaN keys and infinite and NaN values, and the cache past the chunk
    NaN: the queries before it give what they give without it."""
    q, k, v, kc, vc = inputs(n, 4, 2, 77)
    clean = prefill_attention(q, k, v, kc.copy(), vc.copy(), begin, 4, 2, D, THETA, cache="f32")[1].reshape(n, -1)
    k[bad], v[bad, ::2], v[bad, 1::2] = np.nan, np.inf, np.nan
    kc[begin + n:], vc[begin + n:] = np.nan, np.nan
    got = run(device, q, k, v, kc, vc, begin, heads=4, kv_heads=2)[1].reshape(n, -1)
    rms = float(np.sqrt(np.mean(clean[:bad].astype(np.float64) ** 2)))
    assert_close(got[:bad].ravel(), clean[:bad].ravel(), 1e-5 * rms, 2e-5, label="rows before the bad one")
    assert not np.isfinite(got[bad:]).any()
