"""Prompts long enough that the chain's fused launches take the GEMM's wide tiles (q|k|v with RoPE on 64 x 128
and 64 x 256, gate|up on 64 x 256 and 128 x 256), against their unfused forms to the bit."""

import os

import numpy as np
import pytest

import oracle
from enargeia_amd import kernels as K
from enargeia_amd.model import Decoder, DeviceModel, ModelConfig, synthetic_model

pytestmark = pytest.mark.gpu

CFG = ModelConfig(layers=1, max_context=2048)


@pytest.fixture(scope="module")
def model():
    return synthetic_model(CFG)


def run(dev, model, count):
    prompt = [int(t) for t in oracle.random_ids(count, 79, CFG.vocab)]
    shape = (CFG.layers, CFG.max_context, CFG.kv_heads * CFG.head_dim)
    dm = DeviceModel(dev, model)
    dec = Decoder(dm)
    try:
        dec.set_prefill_chunk(CFG.max_context)
        token = dec.prefill(0, prompt)
        caches = [dev.read_array(c, np.uint16, int(np.prod(shape))).reshape(shape)[:, :count]
                  for c in (dec.buffers.k_cache, dec.buffers.v_cache)]
        return token, dec.logits().copy().view(np.uint32), *caches
    finally:
        dec.close()
        dm.release()


@pytest.mark.parametrize("count", [700, 1100, 2048])
def test_wide_tiles_fused_as_unfused(device, model, count):
    token, logits, k, v = run(device, model, count)
    for switch in ("EG_PREFILL_PAIR", "EG_PREFILL_ROPE", "EG_PREFILL_XB16", "EG_PREFILL_XCD"):
        os.environ[switch] = "0"
        try:
            other = K.Device(0)
        finally:
            del os.environ[switch]
        try:
            got = run(other, model, count)
        finally:
            other.close()
        assert got[0] == token, switch
        for a, b in zip(got[1:], (logits, k, v)):
            np.testing.assert_array_equal(a, b, err_msg=switch)
