"""Rows past 256 16-byte chunks (K > 8192 int4, K > 4096 int8): x in LDS, one wave per one or two
rows. Edges: one chunk past the register kernels, the longest row, rows past it (per element), one row,
an odd last pair where rows outnumber the resident waves, bias and outOffset, both encodings."""

import numpy as np
import pytest

import oracle
from conftest import FP32_TOLERANCE, assert_close, gemv_tolerance
from test_gpu_gemv import run_decode

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,k,bits,fmt,bs", [
    (1, 8224, 4, "sym", 32), (6, 8256, 4, "ref", 64), (1001, 11008, 4, "ref", 64), (33, 15360, 4, "sym", 32),
    (7, 15392, 4, "sym", 32), (5, 4112, 8, "sym", 16), (40, 15360, 8, "ref", 64), (3, 12288, 4, "sym", 96),
    (4097, 8256, 4, "ref", 64), (4099, 4160, 8, "sym", 64),
])
def test_longest_rows_match_the_oracle(device, n, k, bits, fmt, bs):
    x = oracle.normal_floats(k, 3000 + k, 1.0)
    w = oracle.normal_floats(n * k, 3100 + n, 0.02)
    q = oracle.quantize_sym(w, n, k, bits, bs) if fmt == "sym" else oracle.quantize_blocks_n(w, n, k, bits, bs)
    bias = oracle.normal_floats(n, 3200 + n, 0.02) if n % 2 else None
    off = 3 if n % 2 else 0
    got = run_decode(device, x, q, bias, out_offset=off)
    expect = oracle.linear_q(x, q, bias, 1)
    assert np.all(got[:off] == 0), "rows before outOffset written"
    tol = FP32_TOLERANCE if fmt == "ref" else gemv_tolerance(expect)
    assert_close(got[off:], expect, *tol, label=f"longest {n}x{k} int{bits} {fmt}")


def test_infinite_input_stays_infinite(device):
    """An infinite x gives infinite sums, as a product per code does, not NaN - from a zero-point's
    share or from a slot past the row's end, which reads x[0..] against zeros."""
    n, k = 9, 8224
    x = np.abs(oracle.normal_floats(k, 5, 1.0))
    q = oracle.quantize_sym(np.full(n * k, 0.5, np.float32), n, k, 4, 32)
    x[0] = np.inf
    assert np.isposinf(run_decode(device, x, q, None)).all()
