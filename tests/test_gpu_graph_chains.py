"""Graphs of a few of the library's kernels in a row, which are launched as those kernels."""
import ctypes

import numpy as np
import pytest

from cogni_ml_amd import hip, quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q6_K

pytestmark = pytest.mark.gpu


def test_graphs_of_a_few_kernels(gpu):
    """A captured chain of the library's kernels (launched as kernels), one with a node of another kind and one too long (launched as graphs):
    the values of the eager calls on every replay, on another stream, after the graph they were made of is gone, with new inputs each time."""
    rng = np.random.default_rng(5)
    tokens, in_dim, out_dim = 3, 512, 300
    w = DevArray(synth.make_weights(rng, Q6_K, out_dim, in_dim))
    x, y, z = DevArray(nbytes=4 * tokens * in_dim), DevArray(nbytes=4 * tokens * out_dim), DevArray(nbytes=4 * tokens * out_dim)
    stream, other = hip.HIPStream(), hip.HIPStream()

    def body(launches, copy):
        s = hip.current_stream_handle()
        for k in range(launches):
            quant.gemv_dev(w.ptr, Q6_K, x.ptr, y.ptr, in_dim, out_dim, tokens, y.ptr if k else 0, s)
        quant.swiglu_dev(y.ptr, y.ptr, z.ptr, tokens * out_dim, s)
        if copy:
            hip.check(hip.lib().hipMemcpyDtoDAsync(ctypes.c_void_p(y.ptr), ctypes.c_void_p(z.ptr), ctypes.c_size_t(4 * tokens * out_dim), s), "copy")

    try:
        for launches, copy in ((1, False), (3, False), (2, True), (8, False)):
            with hip.with_stream(stream):
                body(launches, copy)
            stream.synchronize()
            stream.begin_capture()
            with hip.with_stream(stream):
                body(launches, copy)
            graph = stream.end_capture()
            ex = graph.instantiate()
            graph.close()
            for r in range(4):
                hip.copy_htod(x.ptr, synth.make_activations(rng, tokens, in_dim), 4 * tokens * in_dim, "x")
                with hip.with_stream(stream):
                    body(launches, copy)
                stream.synchronize()
                want = y.read(np.float32, tokens * out_dim), z.read(np.float32, tokens * out_dim)
                hip.copy_htod(z.ptr, np.zeros(tokens * out_dim, np.float32), 4 * tokens * out_dim, "z")
                on = other if r == 2 else stream
                ex.launch(on)
                on.synchronize()
                assert np.array_equal(y.read(np.float32, tokens * out_dim), want[0]) and np.array_equal(z.read(np.float32, tokens * out_dim), want[1])
            ex.close()
    finally:
        for a in (w, x, y, z):
            a.close()
        stream.close()
        other.close()
