"""The f32 cache's attention over chunks that end within two key tiles, where a tile of no more than 16 keys takes
the products of those alone."""

import numpy as np
import pytest

from conftest import assert_close
from oracle.decode import prefill_attention
from test_gpu_prefill_attention import D, THETA, run
from test_gpu_prefill_attention_edges import inputs

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("begin,n,heads,kv_heads", [(0, 2, 16, 8), (0, 16, 14, 2), (0, 17, 14, 2), (64, 16, 8, 8),
                                                     (60, 20, 14, 2), (60, 21, 14, 2), (112, 16, 3, 3), (113, 16, 3, 3)])
def test_few_keys_in_the_last_tile(device, begin, n, heads, kv_heads):
    q, k, v, kc, vc = inputs(n, heads, kv_heads, 7 + begin + n)
    got = run(device, q, k, v, kc.copy(), vc.copy(), begin, heads=heads, kv_heads=kv_heads)[1]
    want = prefill_attention(q, k, v, kc, vc, begin, heads, kv_heads, D, THETA, cache="f32")[1]
    rms = float(np.sqrt(np.mean(want.astype(np.float64) ** 2)))
    assert_close(got.ravel(), want.ravel(), 1e-5 * rms, 2e-5, label=f"begin {begin} n {n} heads {heads}/{kv_heads}")


def test_few_keys_with_an_infinite_one(device):
    """Row 5 of 10 holds NaN keys and infinite and NaN values: the queries before it do not see it."""
    q, k, v, kc, vc = inputs(10, 4, 2, 78)
    clean = prefill_attention(q, k, v, kc.copy(), vc.copy(), 0, 4, 2, D, THETA, cache="f32")[1].reshape(10, -1)
    k[5], v[5, ::2], v[5, 1::2] = np.nan, np.inf, np.nan
    kc[10:], vc[10:] = np.nan, np.nan
    got = run(device, q, k, v, kc, vc, 0, heads=4, kv_heads=2)[1].reshape(10, -1)
    rms = float(np.sqrt(np.mean(clean[:5].astype(np.float64) ** 2)))
    assert_close(got[:5].ravel(), clean[:5].ravel(), 1e-5 * rms, 2e-5, label="rows before the bad one")
    assert not np.isfinite(got[5:]).any()
