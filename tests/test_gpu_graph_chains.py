"""Graphs of a few of the library's kernels in a row, which are launched as those kernels."""
import ctypes

import numpy as np
import pytest

from cogni_ml_amd import hip, quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q6_K

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
            assert hip.lib().mlhip_graph_exec_kernels(ex._handle) == (launches + 1 if launches < 5 and not copy else 0)
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
            handle = ex._handle
            ex.close()
            assert hip.lib().mlhip_graph_exec_kernels(handle) == 0
    finally:
        for a in (w, x, y, z):
            a.close()
        stream.close()
        other.close()


class Layer:
    """A matrix, its input and output, and the operators on them that the tests below capture. `image`: of the packed activations, its own or another layer's."""

    def __init__(self, seed, image=None, tokens=8, in_dim=2048, out_dim=192):
        rng = np.random.default_rng(seed)
        self.shape = in_dim, out_dim, tokens
        self.image = image or DevArray(nbytes=quant.gemv_image_bytes(Q4_K, in_dim, tokens))
        self.x = synth.make_activations(rng, tokens, in_dim)
        self.w, self.xd, self.y = DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)), DevArray(self.x), DevArray(nbytes=4 * tokens * out_dim)

    def gemv(self, residual=False):   # (two kernels)
        st, (in_dim, out_dim, tokens) = hip.current_stream_handle(), self.shape
        quant.gemv_pack_dev(self.xd.ptr, Q4_K, in_dim, tokens, self.image.ptr, st)
        quant.gemv_packed_dev([self.w.ptr], Q4_K, self.image.ptr, [self.y.ptr], [out_dim], in_dim, tokens, self.y.ptr if residual else 0, st)

    def swiglu(self):
        quant.swiglu_dev(self.y.ptr, self.y.ptr, self.y.ptr, self.shape[1] * self.shape[2], hip.current_stream_handle())

    def read(self):
        return self.y.read(np.uint32, self.shape[1] * self.shape[2])

    def close(self):
        for a in (self.w, self.xd, self.y, self.image):
            a.close()


def captured(stream, body, flags=0):
    stream.begin_capture()
    with hip.with_stream(stream):
        body()
    graph = stream.end_capture()
    handle = ctypes.c_void_p()
    hip.check(hip.lib().mlhip_graph_instantiate(ctypes.byref(handle), graph._handle, ctypes.c_uint64(flags)), "instantiate")
    graph.close()
    return hip.HIPGraphExec(handle)


def wait(stream, after):
    """What is enqueued on `stream` from now on waits for what `after` has been given."""
    e = hip.Event()
    e.record(after)
    hip.check(hip.lib().hipStreamWaitEvent(stream.handle, e.handle, ctypes.c_uint(0)), "hipStreamWaitEvent")
    return e


def test_what_is_no_chain_goes_as_a_graph(gpu):
    """Branches, nodes that do not depend on each other, another module's kernel, instantiation flags, and chains that the library has been told to forget: not
    launched as kernels, and the values of the same work in order."""
    a, b = Layer(1), Layer(2)
    s, t = hip.HIPStream(), hip.HIPStream()
    module, events = hip.HIPModule.load_builtin(), []
    n = a.shape[1] * a.shape[2]

    def forked():   # a's product; both products' SwiGLU beside each other; a again
        a.gemv()
        events.append(wait(t, s))
        with hip.with_stream(t):
            b.gemv()
        a.swiglu()
        events.append(wait(s, t))
        a.swiglu()

    def apart():
        events.append(wait(t, s))
        with hip.with_stream(t):
            b.swiglu()
        a.swiglu()
        events.append(wait(s, t))

    def foreign():
        a.gemv()
        params = hip.KernelParams(*[ctypes.c_uint64(a.y.ptr)] * 3, ctypes.c_uint32(n))
        hip.launch(module.function("swiglu_f32"), (n + 255) // 256, 1, 1, 256, 1, 1, params, "swiglu_f32")

    def chain():
        a.gemv()
        a.swiglu()

    try:
        with hip.with_stream(s):   # the values, in order on one stream
            a.gemv(), a.swiglu(), b.gemv()
        s.synchronize()
        once, b0 = a.read(), b.read()
        with hip.with_stream(s):
            a.swiglu()
        s.synchronize()
        twice = a.read()
        for body, flags, want_a, want_b in ((forked, 0, twice, b0), (foreign, 0, once, b0), (chain, 1, once, b0), (apart, 0, None, None)):
            ex = captured(s, body, flags)
            assert hip.lib().mlhip_graph_exec_kernels(ex._handle) == 0, body.__name__
            for _ in range(3):
                if body is apart:   # in place: from the products each time
                    with hip.with_stream(s):
                        a.gemv(), b.gemv()
                    want_a = once
                ex.launch(s)
                s.synchronize()
                assert np.array_equal(a.read(), want_a), body.__name__
                assert want_b is None or np.array_equal(b.read(), want_b), body.__name__
            ex.close()
        ex = captured(s, chain)
        assert hip.lib().mlhip_graph_exec_kernels(ex._handle) == 3
        hip.lib().cogni_internal_drop_chains()
        assert hip.lib().mlhip_graph_exec_kernels(ex._handle) == 0
        ex.launch(s)
        s.synchronize()
        assert np.array_equal(a.read(), once)
        ex.close()
    finally:
        for o in [a, b, module, s, t] + events:
            o.close()


def test_chains_on_a_capturing_stream_become_part_of_that_graph(gpu):
    a, s, t = Layer(3), hip.HIPStream(), hip.HIPStream()
    try:
        inner = captured(s, lambda: (a.gemv(), a.swiglu()))
        with hip.with_stream(s):
            a.gemv(), a.swiglu()
        s.synchronize()
        want = a.read()
        outer = captured(t, lambda: (inner.launch(t), None))
        inner.close()
        for _ in range(3):
            hip.copy_htod(a.y.ptr, np.zeros(a.y.nbytes, np.uint8), a.y.nbytes, "y")
            outer.launch(t)
            t.synchronize()
            assert np.array_equal(a.read(), want)
        outer.close()
    finally:
        for o in (a, s, t):
            o.close()


def test_graphs_that_threads_launch_on_one_stream_follow_each_other_whole(gpu):
    """Chains whose kernels hand data on in one activation image, as multi-token calls on a stream do: one thread's pack between another's pack and product would
    give that one the wrong activations."""
    import threading
    first = Layer(4)
    layers, s = [first, Layer(5, first.image), Layer(6, first.image)], hip.HIPStream()
    try:
        execs = [captured(s, lambda l=l: (l.gemv(), l.gemv(True))) for l in layers]
        assert [hip.lib().mlhip_graph_exec_kernels(e._handle) for e in execs] == [4] * 3
        want = []
        for l in layers:
            with hip.with_stream(s):
                l.gemv(), l.gemv(True)
            s.synchronize()
            want.append(l.read())
        for _ in range(15):
            threads = [threading.Thread(target=lambda e=e: [e.launch(s) for _ in range(20)]) for e in execs]
            for t in threads:
                t.start()
            for t in threads:
                t.join()
            s.synchronize()
            for l, v in zip(layers, want):
                assert np.array_equal(l.read(), v)
        for e in execs:
            e.close()
    finally:
        for o in layers + [s]:
            o.close()
