"""Session set-up shared by the GPU parity tests (all of them call through libcogni_hip.so)."""
import ctypes

import numpy as np
import pytest

from cogni_ml_amd import hip, quant


@pytest.fixture(scope="session")
def gpu():
    ctx = hip.Context.create(0)
    assert ctx.arch.startswith("gfx950"), ctx.arch
    quant.init(0)
    yield ctx
    ctx.close()


class DevArray:
    """A numpy array mirrored into a DeviceBuffer."""

    def __init__(self, host=None, nbytes=None):
        if host is not None:
            host = np.ascontiguousarray(host)
            nbytes = host.nbytes
        self.buf = hip.DeviceBuffer(nbytes)
        self.ptr, self.nbytes = self.buf.ptr, nbytes
        if host is not None and nbytes:
            hip.copy_htod(self.ptr, host, nbytes, "test input")

    def read(self, dtype, count):
        out = np.empty(count, dtype=dtype)
        hip.synchronize()
        hip.copy_dtoh(out, self.ptr, out.nbytes, "test output")
        return out

    def close(self):
        self.buf.close()


def launched_blocks(issue):
    """Workgroup sizes (x) of the kernels that issue(stream handle) launches, in no particular order: captured, not run."""
    L, stream = hip.lib(), hip.HIPStream()
    stream.begin_capture()
    try:
        issue(stream.handle)
    finally:
        graph = stream.end_capture()
    count = ctypes.c_size_t(0)
    hip.check(L.hipGraphGetNodes(graph._handle, None, ctypes.byref(count)), "hipGraphGetNodes")
    nodes = (ctypes.c_void_p * count.value)()
    hip.check(L.hipGraphGetNodes(graph._handle, nodes, ctypes.byref(count)), "hipGraphGetNodes")
    blocks = []
    for node in nodes:
        params = (ctypes.c_uint32 * 64)()   # hipKernelNodeParams, which starts with the block's dimensions
        hip.check(L.hipGraphKernelNodeGetParams(ctypes.c_void_p(node), params), "hipGraphKernelNodeGetParams")
        blocks.append(params[0])
    graph.close()
    stream.close()
    return blocks
