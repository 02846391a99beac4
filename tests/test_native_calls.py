"""cogni_ml_amd._calls: the library gets from a native call exactly what the Python function of that name hands it, and whatever the
native call does not take goes through that function."""
import ctypes
import inspect

import pytest

from cogni_ml_amd import hip, quant
from cogni_ml_amd.types import TensorType

calls = hip.calls
native = pytest.mark.skipif(calls is None, reason="no Python headers when the library was built")

U64, U32 = ctypes.c_uint64, ctypes.c_uint32
PROTO = {"matmul_dev": ctypes.CFUNCTYPE(ctypes.c_int, U64, U32, U64, U64, U64, U32, U32, U32, U64, ctypes.c_size_t, ctypes.c_void_p),
         "gemv_dev": ctypes.CFUNCTYPE(ctypes.c_int, U64, U32, U64, U64, U64, U32, U32, U32, ctypes.c_void_p),
         "dequantize_dev": ctypes.CFUNCTYPE(ctypes.c_int, U64, U32, U64, U64, ctypes.c_void_p)}
BIG = (1 << 64) - 1


class Took(Exception):
    pass


@pytest.fixture
def seen():
    """The library's entry points replaced by ones that note their arguments; the Python functions by ones that say they were called."""
    log, status = [], [0]

    def entry(name):
        def f(*a):
            log.append((name,) + a)
            return status[0]
        return PROTO[name](f)

    def slow(name):
        def f(*a, **k):
            raise Took(name)
        return f

    def check(code):
        raise quant.QuantError(code)

    kept = [entry(n) for n in PROTO]
    hip.lib()
    calls.set_python(*(slow(n) for n in PROTO), check, TensorType, ctypes.c_void_p)
    calls.set_library(*(ctypes.cast(f, ctypes.c_void_p).value for f in kept))
    yield log, status
    L = hip.lib()
    calls.set_python(*(getattr(quant, "_%s" % n) for n in PROTO), quant._check, TensorType, ctypes.c_void_p)
    calls.set_library(*(ctypes.cast(f, ctypes.c_void_p).value for f in (L.cogni_matmul_dev, L.cogni_gemv_dev, L.cogni_dequantize_dev)))


@native
@pytest.mark.parametrize("stream,want", [(None, None), (0, None), (0x7F0012345678, 0x7F0012345678), (ctypes.c_void_p(), None),
                                         (ctypes.c_void_p(0x7F0012345678), 0x7F0012345678)])
def test_arguments_arrive_where_the_python_functions_put_them(seen, stream, want):
    log, _ = seen
    calls.matmul_dev(1, TensorType.Q8_0, 2, 3, 4, 5, 6, 7, 8, 9, stream)
    calls.matmul_dev(BIG, 12, 2, 3, 4, 5, 0xFFFFFFFF, stream=stream, bias_ptr=9)
    calls.matmul_dev(out_ptr=3, w_ptr=1, w_type=8, tokens=6, x_ptr=2, out_dim=5, in_dim=4, workspace_bytes=8, workspace_ptr=7, stream=stream)
    calls.gemv_dev(1, TensorType.Q6_K, 2, 3, 4, 5, stream=stream)
    calls.gemv_dev(1, 14, 2, 3, 4, 5, 6, 7, stream)
    calls.dequantize_dev(1, TensorType.F16, 2, 3, stream)
    calls.dequantize_dev(1, 1, BIG, out_ptr=3, stream=stream)
    assert log == [("matmul_dev", 1, 8, 2, 9, 3, 4, 5, 6, 7, 8, want), ("matmul_dev", BIG, 12, 2, 9, 3, 4, 5, 0xFFFFFFFF, 0, 0, want),
                   ("matmul_dev", 1, 8, 2, 0, 3, 4, 5, 6, 7, 8, want), ("gemv_dev", 1, 14, 2, 0, 3, 4, 5, 1, want),
                   ("gemv_dev", 1, 14, 2, 7, 3, 4, 5, 6, want), ("dequantize_dev", 1, 1, 2, 3, want), ("dequantize_dev", 1, 1, BIG, 3, want)]


@native
@pytest.mark.parametrize("args,kw", [((1, 8, 2, 3, 4, 5), {}), ((1, 8, 2, 3, 4, 5, -1), {}), ((1 << 64, 8, 2, 3, 4, 5, 6), {}),
                                     ((1, 8, 2, 3, 4, 5, 1 << 32), {}), ((1, -8, 2, 3, 4, 5, 6), {}), ((1.0, 8, 2, 3, 4, 5, 6), {}),
                                     ((1, "8", 2, 3, 4, 5, 6), {}), ((None, 8, 2, 3, 4, 5, 6), {}), ((True, 8, 2, 3, 4, 5, 6), {}),
                                     ((1, 8, 2, 3, 4, 5, 6), {"tokens": 6}), ((1, 8, 2, 3, 4, 5, 6), {"nothing": 1}),
                                     ((1, 8, 2, 3, 4, 5, 6, 7, 8, 9, None, 10), {}), ((1, 8, 2, 3, 4, 5, ctypes.c_uint32(6)), {}),
                                     ((1, 8, 2, 3, 4, 5, 6), {"stream": ctypes.c_uint64(5)}), ((1, 8, 2, 3, 4, 5, 6), {"stream": True}),
                                     ((1, 8, 2, 3, 4, 5, 6), {"stream": -1})])
def test_other_calls_go_to_the_python_function(seen, args, kw):
    log, _ = seen
    with pytest.raises(Took, match="matmul_dev"):
        calls.matmul_dev(*args, **kw)
    assert log == []


@native
def test_a_status_raises_what_check_raises(seen):
    log, status = seen
    status[0] = -3
    for f, args in ((calls.matmul_dev, (1, 8, 2, 3, 4, 5, 6)), (calls.gemv_dev, (1, 8, 2, 3, 4, 5)), (calls.dequantize_dev, (1, 8, 2, 3))):
        with pytest.raises(quant.QuantError) as e:
            f(*args)
        assert e.value.code == -3
    assert len(log) == 3


@native
def test_signatures_are_those_of_the_python_functions():
    for n in PROTO:
        assert inspect.signature(getattr(quant, n)) == inspect.signature(getattr(quant, "_%s" % n))


class FakeLib:
    def __init__(self):
        self.log, self.status = [], 0

    def cogni_a_dev(self, *args):
        self.log.append(("a",) + args)
        return self.status

    def cogni_b_dev(self, *args):
        self.log.append(("b",) + args)
        return self.status

    def cogni_rule(self, *args):
        self.log.append(("rule",) + args)
        return 7


def test_a_sequence_is_issued_again_with_the_same_calls(monkeypatch):
    """hip.issue: operators alone are kept, on whatever stream is current, per key and per owner; errors raise; another thread that
    calls the library meanwhile is not noted."""
    import threading
    fake = FakeLib()
    monkeypatch.setattr(hip, "_lib", fake)
    stream = type("S", (), {"handle": "s1"})()
    raised = []

    def launch():
        n = hip.lib().cogni_rule(5)
        hip.lib().cogni_a_dev(1, n, hip.current_stream_handle())
        t = threading.Thread(target=lambda: hip.lib().cogni_b_dev(99, None))
        t.start()
        t.join()
        hip.lib().cogni_b_dev(2, hip.current_stream_handle())

    kept = {}
    for _ in range(2):   # as it is written; the same, noted
        hip.issue(kept, 3, launch, raised.append)
        assert fake.log == [("rule", 5), ("a", 1, 7, None), ("b", 99, None), ("b", 2, None)] and hip.lib() is fake
        fake.log.clear()
    with hip.with_stream(stream):
        hip.issue(kept, 3, launch, raised.append)
    assert fake.log == [("a", 1, 7, "s1"), ("b", 2, "s1")] and raised == []
    fake.log.clear()
    hip.issue(kept, 4, launch, raised.append)
    assert fake.log[0] == ("rule", 5) and sorted(kept) == [3, 4]
    fake.status = -2
    with pytest.raises(ZeroDivisionError):
        hip.issue(kept, 3, launch, lambda code: 1 // 0)

    def fails():
        hip.lib().cogni_a_dev(1, None)
        raise KeyError("no")
    fake.status = 0
    with pytest.raises(KeyError):
        hip.issue(kept, 5, fails, raised.append)
    assert 5 not in kept
    hip.issue(kept, 5, launch, raised.append)
    with pytest.raises(KeyError):
        hip.issue(kept, 5, fails, raised.append)
    assert not kept[5] and hip.lib() is fake
    for k in range(200):
        hip.issue(kept, 100 + k // 2, launch, raised.append)
    assert len(kept) <= 32


class OtherLib(FakeLib):
    """FakeLib with the entry points of the single-operator calls, a call of the driver layer and one that sets something."""

    def _note(name):
        return lambda self, *args: (self.log.append((name,) + args), self.status)[1]

    typed_matmul_dev, typed_gemv_dev, typed_dequantize_dev = _note("matmul"), _note("gemv"), _note("dequantize")
    mlhip_memcpy_dtod, cogni_set_gemm_threshold, cogni_matmul_add, cogni_gemm_tall_takes = _note("copy"), _note("set"), _note("host"), _note("takes")


@pytest.fixture
def other(monkeypatch):
    """The library replaced by an OtherLib, for the native calls as well."""
    hip.lib()
    fake = OtherLib()
    monkeypatch.setattr(hip, "_lib", fake)
    if calls is not None:
        kept = [PROTO[n](lambda *a, n=n: (fake.log.append((n[:-4],) + a), 0)[1]) for n in ("matmul_dev", "gemv_dev", "dequantize_dev")]
        calls.set_library(*(ctypes.cast(f, ctypes.c_void_p).value for f in kept))
    yield fake
    monkeypatch.undo()
    if calls is not None:
        L = hip.lib()
        calls.set_library(*(ctypes.cast(f, ctypes.c_void_p).value for f in (L.cogni_matmul_dev, L.cogni_gemv_dev, L.cogni_dequantize_dev)))


def passes(fake, kept, key, launch, count=4):
    """What the library is called with, pass by pass."""
    out = []
    for _ in range(count):
        hip.issue(kept, key, launch, lambda code: None)
        out.append(list(fake.log))
        fake.log.clear()
    return out


def test_single_operator_calls_are_part_of_a_noted_sequence(other):
    def launch():
        st = hip.current_stream_handle()
        quant.dequantize_dev(1, TensorType.Q4_K, 2, 3, st)
        hip.lib().cogni_a_dev(4, st)
        quant.matmul_dev(1, 12, 2, 3, 4, 5, 6, 7, 8, 9, st)
        quant.gemv_dev(1, 14, 2, 3, 4, 5, stream=st)

    want = [("dequantize", 1, 12, 2, 3, None), ("a", 4, None), ("matmul", 1, 12, 2, 9, 3, 4, 5, 6, 7, 8, None), ("gemv", 1, 14, 2, 0, 3, 4, 5, 1, None)]
    kept = {}
    assert passes(other, kept, 1, launch) == [want] * 4 and len(kept[1]) == 4


@pytest.mark.parametrize("what", [lambda: hip.lib().mlhip_memcpy_dtod(1, 2, 3), lambda: hip.lib().cogni_set_gemm_threshold(4), lambda: hip.lib().cogni_matmul_add(5),
                                  lambda: hip.lib().cogni_b_dev(6, 0x1234), lambda: hip.lib().cogni_b_dev()])
def test_what_is_no_operator_on_the_current_stream_is_done_every_time(other, what):
    """Copies, settings, operators on host arrays or on another stream: such a sequence is launched as it is written, whatever else it does."""
    def launch():
        hip.lib().cogni_gemm_tall_takes(1)
        hip.lib().cogni_a_dev(2, hip.current_stream_handle())
        what()

    kept = {}
    first, *rest = passes(other, kept, 1, launch)
    assert len(first) == 3 and rest == [first] * 3 and kept[1] is False


def test_a_sequence_within_a_sequence(other):
    inner, outer, stream = {}, {}, type("S", (), {"handle": "s1"})()

    def launch_inner():
        hip.lib().cogni_a_dev(1, hip.current_stream_handle())

    def launch():
        hip.issue(inner, 1, launch_inner, lambda code: None)
        hip.lib().cogni_b_dev(2, hip.current_stream_handle())

    for _ in range(3):
        hip.issue(inner, 1, launch_inner, lambda code: None)
    other.log.clear()
    with hip.with_stream(stream):
        assert passes(other, outer, 1, launch) == [[("a", 1, "s1"), ("b", 2, "s1")]] * 4
    assert len(outer[1]) == 2


def test_the_oldest_notes_go_first(other):
    kept = {}

    def launch():
        hip.lib().cogni_gemm_tall_takes(1)
        hip.lib().cogni_a_dev(2, hip.current_stream_handle())

    for key in range(40):
        passes(other, kept, key, launch, 2)
    assert sorted(kept) == list(range(8, 40)) and all(len(kept[k]) == 1 for k in kept)
    assert passes(other, kept, 8, launch, 1) == [[("a", 2, None)]]


def test_threads_note_their_own_calls(other):
    import threading
    kept, go = [{} for _ in range(4)], threading.Barrier(4)

    def work(i):
        def launch():
            go.wait()
            for k in range(50):
                hip.lib().cogni_a_dev(100 * i + k, hip.current_stream_handle())
            go.wait()
        for _ in range(2):
            hip.issue(kept[i], "k", launch, lambda code: None)

    threads = [threading.Thread(target=work, args=(i,)) for i in range(4)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    for i in range(4):
        assert [a for f, a in kept[i]["k"]] == [(100 * i + k,) for k in range(50)]
    assert hip.lib() is other
