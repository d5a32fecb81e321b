"""A chunk of more query blocks than a grid's y takes (65535), in as many launches as it needs: recorded into a
graph that is never launched (its attention would take seconds)."""

import ctypes

import pytest

from enargeia_amd import _lib
from enargeia_amd import kernels as K
from test_gpu_prefill_attention import D, THETA, PrefillDims

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("entry", ["eg_attention_prefill", "eg_attention_prefill_f32"])
def test_more_query_blocks_than_a_grid_takes(entry):
    queries = 65535 * 64 + 1
    dev = K.Device(0)
    buf = dev.buffer(1 << 12)
    try:
        d = PrefillDims(queries, queries, 0, 1, 1, D, queries, THETA)
        dev.capture_begin()
        _lib.check(getattr(_lib.load(), entry)(dev.ctx, *[ctypes.c_void_p(buf.ptr)] * 7, ctypes.byref(d)), dev.ctx)
        graph = dev.capture_end()
        hip, count = _lib.load(), ctypes.c_size_t()
        handle = ctypes.cast(graph.handle, ctypes.POINTER(ctypes.c_void_p))[0]  # eg_graph's first member
        assert hip.hipGraphGetNodes(ctypes.c_void_p(handle), None, ctypes.byref(count)) == 0
        assert count.value == 3  # RoPE and append, two attention launches
        graph.destroy()
    finally:
        buf.release()
        dev.close()
