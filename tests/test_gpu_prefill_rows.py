"""The prefill GEMM's bf16 rows of f32 x: where the tile wants them they are held in the buffer
that the context was created with, a stretch of rows at a time, and calls that may not use it - under a
capture, on a caller's stream - stage the f32 rows themselves with the same sums, to the bit."""

import ctypes
import os

import numpy as np
import pytest

import oracle
from conftest import assert_close
from enargeia_amd import _lib
from enargeia_amd import kernels as K
from test_gpu_prefill import model_tol, run_prefill, run_swiglu

pytestmark = pytest.mark.gpu


def device_with(tile):
    """A context whose prefill GEMMs take `tile`."""
    os.environ["EG_PREFILL_TILE"] = tile
    try:
        return K.Device(0)
    finally:
        del os.environ["EG_PREFILL_TILE"]


class Gemm:
    """One prefill projection bound to its buffers."""

    def __init__(self, dev, m, n, k, bits=4, seed=1):
        self.dev, self.m, self.n = dev, m, n
        w = oracle.normal_floats(n * k, seed, 0.02)
        self.q = oracle.quantize_sym(w, n, k, bits, 32)
        self.x = dev.buffer(m * k * 4)
        self.w = [dev.upload(self.q.packed), dev.upload(self.q.scales)]
        self.out = dev.buffer(m * n * 4)
        self.kern = K.ComputeKernel(dev, K.with_format(K.MATMUL_Q4_PREFILL, bits, self.q.encoding))
        u = self.kern.uniform()
        u.write(K.matmul_q4_dims(m, n, k, False, 32))
        self.group = self.kern.bind_group([self.x, *self.w, None, None, self.out, u])

    def set_x(self, x):
        self.dev.write(self.x, x)
        self.dev.sync()

    def encode(self):
        self.kern.encode(self.group, K.matmul_q4_prefill_workgroups(self.m, self.n))

    def read(self):
        return self.dev.read_array(self.out, np.uint32, self.m * self.n)

    def release(self):
        for b in [self.x, *self.w, self.out]:
            b.release()


# The tiles that take bf16 rows, each at a ragged shape of several chunks per K group, both code widths.
TILES = [("128,2,2,4", 100, 200, 1120, 4), ("128,4,2,2", 200, 196, 736, 4), ("128,4,4,1", 200, 300, 416, 4),
         ("128,4,2,2", 130, 130, 672, 8)]


@pytest.mark.parametrize("tile,m,n,k,bits", TILES)
def test_a_captured_call_equals_an_eager_one(tile, m, n, k, bits):
    dev = device_with(tile)
    g = Gemm(dev, m, n, k, bits)
    other = Gemm(dev, 300, 260, 416, seed=5)  # eager work between the replays
    try:
        xs = [oracle.normal_floats(m * k, 20 + i, 1.0) for i in range(3)]
        other.set_x(oracle.normal_floats(300 * 416, 9, 1.0))
        g.set_x(xs[0])
        dev.capture_begin()
        g.encode()
        graph = dev.capture_end()
        for x in xs:
            g.set_x(x)
            g.encode()
            eager = g.read()
            model = oracle.linear_q_bf16_fast(x, g.q, None, m)
            assert_close(eager.view(np.float32), model, *model_tol(model), label=f"eager {tile}")
            other.encode()
            dev.zero(g.out, m * n * 4)
            graph.launch()
            other.encode()
            np.testing.assert_array_equal(g.read(), eager)
        graph.destroy()
    finally:
        g.release()
        other.release()
        dev.close()


@pytest.mark.parametrize("tile,m,n,k,bits", TILES)
def test_a_callers_stream_gives_the_same_bits(tile, m, n, k, bits):
    dev, owner = device_with(tile), K.Device(0)
    g = Gemm(dev, m, n, k, bits)
    try:
        g.set_x(oracle.normal_floats(m * k, 3, 1.0))
        g.encode()
        own = g.read()
        dev.zero(g.out, m * n * 4)
        dev.sync()
        _lib.check(_lib.load().eg_set_stream(dev.ctx, ctypes.c_void_p(owner.stream)), dev.ctx)
        g.encode()
        np.testing.assert_array_equal(g.read(), own)
        _lib.check(_lib.load().eg_set_stream(dev.ctx, None), dev.ctx)
    finally:
        g.release()
        dev.close()
        owner.close()


def test_rows_past_the_buffer():
    """4500 rows of 8192 are 70 MiB as bf16: two stretches, the same bits as two calls."""
    m, n, k, half = 4500, 200, 8192, 2250
    dev = device_with("128,4,2,2,1")
    x = np.tile(oracle.normal_floats(90 * k, 4, 1.0), 50)
    x = (x.reshape(m, k) * np.linspace(0.5, 1.5, m, dtype=np.float32)[:, None]).astype(np.float32)
    q = oracle.quantize_sym(oracle.normal_floats(n * k, 8, 0.02), n, k, 4, 32)
    bias = oracle.normal_floats(n, 3, 0.02)
    try:
        whole = run_prefill(dev, x.reshape(-1), q, bias, m, out_stride=n + 4, out_len=m * (n + 4)).reshape(m, n + 4)
        assert not whole[:, n:].any()
        for at in (0, half):
            part = run_prefill(dev, x[at:at + half].reshape(-1), q, bias, half).reshape(half, n)
            np.testing.assert_array_equal(whole[at:at + half, :n].view(np.uint32), part.view(np.uint32))
        last = oracle.linear_q_bf16_fast(x[-20:].reshape(-1), q, bias, 20)
        assert_close(whole[-20:, :n].ravel(), last, *model_tol(last), label="last rows")
    finally:
        dev.close()


def test_calls_in_a_row_go_round_the_buffer():
    """Ten calls of 16 MiB of rows, none waited for: each gives what it gives alone."""
    m, n, k = 2048, 130, 4096
    dev = device_with("128,4,2,2,1")
    calls = [Gemm(dev, m, n, k) for _ in range(10)]
    try:
        base = oracle.normal_floats(m * k, 6, 1.0)
        for i, g in enumerate(calls):
            g.set_x(np.roll(base, 977 * i))
        for g in calls:
            g.encode()
        got = [g.read() for g in calls]
        for g, y in zip(calls, got):
            g.encode()
            np.testing.assert_array_equal(g.read(), y)
        for i in (0, 9):
            model = oracle.linear_q_bf16_fast(np.roll(base, 977 * i)[:40 * k], calls[i].q, None, 40)
            assert_close(got[i].view(np.float32)[:40 * n], model, *model_tol(model), label=f"call {i}")
    finally:
        for g in calls:
            g.release()
        dev.close()


def test_a_call_allocates_nothing():
    """The free device memory is the same before and after a context's first wide call."""
    lib = _lib.load()
    dev = K.Device(0)
    g = Gemm(dev, 2048, 4096, 1024)
    free, total = ctypes.c_size_t(), ctypes.c_size_t()

    def free_bytes():
        dev.sync()
        assert lib.hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
        return free.value

    try:
        # (a small call first: the runtime's own allocations for the first kernels are not meant)
        small = Gemm(dev, 4, 64, 64)
        small.set_x(np.zeros(4 * 64, np.float32))
        small.encode()
        g.set_x(np.ones(2048 * 1024, np.float32))
        before = free_bytes()
        for _ in range(3):
            g.encode()
        assert free_bytes() == before
        small.release()
    finally:
        g.release()
        dev.close()


def test_one_launch_swiglu_leaves_its_scratch_alone(device):
    """K up to 1984 takes one launch, which does not use the scratch rows, whatever tile it takes."""
    m, n, k = 1030, 4172, 160
    x = oracle.normal_floats(m * k, 2, 1.0)
    gate, up = (oracle.quantize_sym(oracle.normal_floats(n * k, s, 0.05), n, k, 4, 32) for s in (3, 4))
    bufs = [device.upload(a) for a in (x, gate.packed, gate.scales, up.packed, up.scales)]
    mark = np.full(2 * n * m, 0x7A5A5A5A, np.uint32)
    out, scratch = device.buffer(m * n * 4), device.upload(mark)
    d = K.MatmulDims.from_buffer_copy(K.matmul_q4_dims(m, n, k, False, 32, n, 0))
    p = [ctypes.c_void_p(b.ptr) for b in bufs]
    try:
        _lib.check(_lib.load().eg_matmul_q4_prefill_swiglu(device.ctx, p[0], p[1], p[2], None, p[3], p[4], None,
                                                           ctypes.c_void_p(out.ptr), ctypes.c_void_p(scratch.ptr),
                                                           ctypes.byref(d), gate.encoding, 4), device.ctx)
        np.testing.assert_array_equal(device.read_array(scratch, np.uint32, mark.size), mark)
        want = run_swiglu(device, x, gate, up, m)
        np.testing.assert_array_equal(device.read_array(out, np.float32, m * n), want)
    finally:
        for b in bufs + [out, scratch]:
            b.release()
