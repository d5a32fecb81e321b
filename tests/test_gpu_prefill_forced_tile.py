"""EG_PREFILL_TILE: one of the prefill GEMM's tiles for every launch that has it, anything else ignored."""

import os

import numpy as np
import pytest

import oracle
from conftest import assert_close
from enargeia_amd import kernels as K
from enargeia_amd.model import Decoder, DeviceModel, ModelConfig, synthetic_model
from test_gpu_prefill import model_tol, run_prefill
from test_gpu_prefill_rows import device_with

pytestmark = pytest.mark.gpu

TILES = ["128,1,1,4", "128,2,1,4", "64,2,2,2", "128,2,2,2", "128,2,2,4", "128,2,4,1", "128,4,2,2", "128,4,4,1", "64,1,1,4",
         "64,2,1,4"]


@pytest.mark.parametrize("value", ["", "64", "128,2,0,1", "128,2,4,0", "0,0,0,0", "128,3,1,4", "32,1,1,4", "128,1,1,4,-2",
                                   "128,1,1,4,1000", "-128,2,1,4", "nonsense"])
def test_what_names_no_tile_is_ignored(device, value):
    m, n, k = 70, 130, 2080
    x = oracle.normal_floats(m * k, 1, 1.0)
    q = oracle.quantize_sym(oracle.normal_floats(n * k, 2, 0.02), n, k, 4, 32)
    dev = device_with(value)
    try:
        np.testing.assert_array_equal(run_prefill(dev, x, q, None, m).view(np.uint32),
                                      run_prefill(device, x, q, None, m).view(np.uint32))
    finally:
        dev.close()


@pytest.mark.parametrize("tile", TILES)
@pytest.mark.parametrize("bits,fmt", [(4, "sym"), (8, "ref")])
def test_blocks_of_16_codes(tile, bits, fmt):
    """A lane of a 128-deep chunk takes two scales for 64 codes: 16-code blocks keep the 64-deep tiles."""
    m, n, k = 70, 200, 416
    x = oracle.normal_floats(m * k, 1, 1.0)
    w = oracle.normal_floats(n * k, 2, 0.02)
    q = oracle.quantize_sym(w, n, k, bits, 16) if fmt == "sym" else oracle.quantize_blocks_n(w, n, k, bits, 16)
    dev = device_with(tile)
    try:
        model = oracle.linear_q_bf16_fast(x, q, None, m)
        assert_close(run_prefill(dev, x, q, None, m), model, *model_tol(model), label=f"{tile} int{bits}")
    finally:
        dev.close()


@pytest.mark.parametrize("tile", TILES)
def test_a_prompt_runs_with_every_tile(device, tile):
    """A prompt short enough that its launches fold the norm, which the wide tiles do not: the logits of
    the library's own choice, at the bar of one bf16 rounding per layer boundary."""
    cfg = ModelConfig(layers=2, max_context=128)
    m = synthetic_model(cfg)
    prompt = [int(t) for t in oracle.random_ids(40, 77, cfg.vocab)]
    got = []
    forced = device_with(tile)
    try:
        for dev in (device, forced):
            dm = DeviceModel(dev, m)
            dec = Decoder(dm)
            try:
                dec.prefill(0, prompt)
                got.append(dec.logits().astype(np.float64))
            finally:
                dec.close()
                dm.release()
    finally:
        forced.close()
    # two layers' bf16 roundings (2^-9 each) of sums in another order
    assert np.linalg.norm(got[1] - got[0]) <= 2e-2 * np.linalg.norm(got[0])
