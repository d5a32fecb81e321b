"""The prefill GEMM's tiles at their edges: rows and columns that do not fill the last tile, K that does
not fill the last chunk, both encodings and both code widths, against the oracle's bf16 model at the
f32 sums' 1e-4 - at shapes for which the library chooses each tile, and with each tile forced."""

import os

import numpy as np
import pytest

import oracle
from conftest import assert_close
from enargeia_amd import kernels as K
from test_gpu_prefill import model_tol, run_prefill, run_swiglu
from test_gpu_prefill_rows import device_with

pytestmark = pytest.mark.gpu


def weights(n, k, bits, fmt, bs):
    v = oracle.normal_floats(n * k, 7 + n + k, 0.02)
    return oracle.quantize_sym(v, n, k, bits, bs) if fmt == "sym" else oracle.quantize_blocks_n(v, n, k, bits, bs)


@pytest.mark.parametrize("m,n,k,bits,fmt,bs", [
    (1, 64, 32, 4, "sym", 32), (33, 100, 160, 4, "sym", 32), (31, 70, 192, 8, "ref", 64),     # 32 x 64 fine
    (300, 2200, 160, 4, "sym", 32), (290, 2250, 192, 8, "sym", 32),                           # 64 x 64 fine
    (330, 3300, 160, 4, "ref", 32),                                                           # 64 x 128
    (300, 3400, 2080, 4, "sym", 32),                                                          # 64 x 128 deep
    (450, 4600, 96, 4, "sym", 32), (450, 4600, 192, 8, "ref", 64),                            # 64 x 256
    (520, 3910, 2080, 4, "ref", 32),                                                          # 128 x 128
    (1030, 4170, 160, 4, "sym", 32), (1030, 4170, 192, 8, "ref", 64),                         # 128 x 256
    (40, 200, 2112, 4, "ref", 64), (20, 96, 4128, 8, "sym", 32),                              # K split over the grid
    (33, 100, 96, 4, "sym", 16), (600, 4600, 96, 4, "ref", 16),                               # blocks of 16
])
def test_tile_edges_match_the_bf16_model(device, m, n, k, bits, fmt, bs):
    x = oracle.normal_floats(m * k, m, 1.0)
    q = weights(n, k, bits, fmt, bs)
    bias = oracle.normal_floats(n, 3, 0.02)
    got = run_prefill(device, x, q, bias, m)
    model = oracle.linear_q_bf16_fast(x, q, bias, m)
    assert_close(got, model, *model_tol(model), label=f"{m}x{n}x{k} int{bits} {fmt} {bs}")


TILES = {"32 x 64 fine": "64,1,1,4", "64 x 64 fine": "64,2,1,4", "32 x 64": "128,1,1,4", "64 x 64": "128,2,1,4",
         "64 x 128": "64,2,2,2", "64 x 128 long": "128,2,2,2", "64 x 128 deep": "128,2,2,4", "64 x 256": "128,2,4,1",
         "128 x 128": "128,4,2,2", "128 x 256": "128,4,4,1"}


@pytest.mark.parametrize("m,n,k,tile", [
    (70, 200, 736, "32 x 64 fine"), (300, 2200, 736, "64 x 64 fine"), (33, 100, 1440, "32 x 64"),
    (290, 1670, 1440, "64 x 64"), (330, 3300, 736, "64 x 128"), (600, 4600, 416, "64 x 256"),
    (1030, 4170, 416, "128 x 256"), (200, 2300, 2112, "32 x 64"), (20, 5000, 4512, "32 x 64"),
    (300, 2200, 2080, "64 x 64"), (100, 1400, 8224, "64 x 128 long"), (300, 3400, 2080, "64 x 128 deep"),
    (520, 3910, 2080, "128 x 128")])
def test_the_library_chooses(device, m, n, k, tile):
    """The library's own choice at a shape of each line of its rule: a launch sums in the order of its
    chunks and K groups, so it equals the tile's forced launch to the bit (K is long enough that the
    other orders differ)."""
    x = oracle.normal_floats(m * k, m, 1.0)
    q = weights(n, k, 4, "sym", 32)
    forced = device_with(TILES[tile])
    try:
        np.testing.assert_array_equal(run_prefill(device, x, q, None, m).view(np.uint32),
                                      run_prefill(forced, x, q, None, m).view(np.uint32))
    finally:
        forced.close()


@pytest.mark.parametrize("tile", list(TILES))
@pytest.mark.parametrize("n", [65, 126, 191, 320])
def test_cut_runs_of_columns(tile, n):
    """n that leaves one, two or three columns of a run of four, or none: every column is stored, and
    nothing past the rows; 70 and 150 rows, the last chunk of K short."""
    k = 416
    dev = device_with(TILES[tile])
    try:
        for m, fmt, bits in ((70, "sym", 4), (150, "ref", 8)):
            x = oracle.normal_floats(m * k, m, 1.0)
            q = weights(n, k, bits, fmt, 32)
            bias = oracle.normal_floats(n, 3, 0.02)
            got = run_prefill(dev, x, q, bias, m, out_len=m * n + 300)
            model = oracle.linear_q_bf16_fast(x, q, bias, m)
            assert_close(got[:m * n], model, *model_tol(model), label=f"{tile} n {n} m {m}")
            assert not got[m * n:].any()
    finally:
        dev.close()


@pytest.mark.parametrize("m,n,k,tile", [
    *((130, 300, 416, TILES[t]) for t in TILES if t not in ("64 x 128 long", "64 x 128 deep", "128 x 128")),
    (600, 4864, 160, None), (1030, 4164, 160, None)])
def test_swiglu_tiles(device, m, n, k, tile):
    """The paired launch with each tile that has one, and at rows for which the library takes the
    64 x 256 and 128 x 256 ones, against gate | up and silu_mul_rows to the bit."""
    x = oracle.normal_floats(m * k, 11, 1.0)
    gate, up = (oracle.quantize_sym(oracle.normal_floats(n * k, s, 0.05), n, k, 4, 32) for s in (12, 13))
    paired = device_with(tile) if tile else device
    os.environ["EG_PREFILL_PAIR"] = "0"
    try:
        apart = device_with(tile or "")
    finally:
        del os.environ["EG_PREFILL_PAIR"]
    try:
        got, want = (run_swiglu(d, x, gate, up, m) for d in (paired, apart))
        np.testing.assert_array_equal(got.view(np.uint32), want.view(np.uint32))
        g, u = (oracle.linear_q_bf16_fast(x, w, None, m).astype(np.float64) for w in (gate, up))
        ref = g / (1 + np.exp(-g)) * u
        assert np.linalg.norm(got - ref) <= 1e-4 * np.linalg.norm(ref)  # f32 sums
    finally:
        apart.close()
        if tile:
            paired.close()


@pytest.mark.parametrize("m,n,k", [(70, 96, 96), (450, 4600, 96), (1030, 4170, 96)])
def test_unaligned_outputs(device, m, n, k):
    """Rows 3 floats longer than n at an odd offset: the outputs take single stores, and nothing
    between the rows is written."""
    x = oracle.normal_floats(m * k, m, 1.0)
    q = weights(n, k, 4, "sym", 32)
    stride, off = n + 3, 1
    got = run_prefill(device, x, q, None, m, out_len=m * stride + off, out_stride=stride, out_offset=off)
    model = oracle.linear_q_bf16_fast(x, q, None, m)
    rows = got[off:].reshape(m, stride)
    assert_close(rows[:, :n].ravel(), model, *model_tol(model), label="offset rows")
    assert not rows[:, n:].any() and got[0] == 0


@pytest.mark.parametrize("m,n,k", [(70, 200, 96), (450, 4600, 160), (1030, 4170, 160)])
def test_nan_rows_stay_in_their_rows(device, m, n, k):
    """A row of NaN next to others, K ending inside a chunk: the zero weights past K meet zeros, not
    the next row's values, so only that row's outputs are NaN."""
    x = oracle.normal_floats(m * k, m, 1.0).reshape(m, k)
    q = weights(n, k, 4, "sym", 32)
    model = oracle.linear_q_bf16_fast(x.reshape(-1), q, None, m).reshape(m, n)
    x[2] = np.nan
    x[m - 1, k - 1] = np.inf
    got = run_prefill(device, x.reshape(-1), q, None, m).reshape(m, n)
    keep = [r for r in range(m) if r not in (2, m - 1)]
    assert np.isnan(got[2]).all() and not np.isfinite(got[m - 1]).all()
    assert_close(got[keep].ravel(), model[keep].ravel(), *model_tol(model), label="rows beside NaN")


def test_bf16_rows_across_streams(device):
    """Launches that take the library's bf16 rows of x on the context's own stream, beside launches of the
    same context on another stream with nothing waiting between them: each reads its own rows."""
    m, n, k = 1030, 4170, 160
    q = weights(n, k, 4, "sym", 32)
    dev = K.Device(0)
    others = [K.Device(0)]  # a second stream to enqueue on
    try:
        kern = K.ComputeKernel(dev, K.with_format(K.MATMUL_Q4_PREFILL, 4, q.encoding))
        w = [dev.upload(q.packed), dev.upload(q.scales)]
        u = kern.uniform()
        u.write(K.matmul_q4_dims(m, n, k, False, q.block_size))
        xs = [oracle.normal_floats(m * k, 50 + i, 1.0) for i in range(8)]
        bx, bo = [dev.upload(x) for x in xs], [dev.buffer(m * n * 4) for _ in xs]
        from enargeia_amd import _lib
        for i in range(8):
            _lib.check(_lib.load().eg_set_stream(dev.ctx, others[0].stream if i % 2 else None), dev.ctx)
            kern.encode(kern.bind_group([bx[i], *w, None, None, bo[i], u]), K.matmul_q4_prefill_workgroups(m, n))
        for o in others:
            o.sync()
        _lib.check(_lib.load().eg_set_stream(dev.ctx, None), dev.ctx)
        for i in (0, 1, 6, 7):
            model = oracle.linear_q_bf16_fast(xs[i], q, None, m)
            assert_close(dev.read_array(bo[i], np.float32, m * n), model, *model_tol(model), label=f"call {i}")
    finally:
        for o in others:
            o.sync()
        dev.close()
        for o in others:
            o.close()
