"""Launches that do the work of several in a layer: each gives, bit for bit, what the separate launches give."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K

pytestmark = pytest.mark.gpu


# resident and streamed operands, next rows that fill their k-slices and that do not, few and all tokens, workgroups that walk
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(4096, 12288, 16), (2048, 256, 9), (1024, 2816, 13), (6144, 2048, 1), (12288, 512, 10)])
def test_swiglu_that_writes_the_next_image(gpu, in_dim, out_dim, tokens):
    rng = np.random.default_rng(in_dim + out_dim + tokens)
    wg, wu = (DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)) for _ in range(2))
    xd = DevArray(synth.make_activations(rng, tokens, in_dim))
    n, nb = tokens * out_dim, quant.gemv_image_bytes(Q6_K, out_dim, 8)
    image = DevArray(nbytes=quant.gemv_image_bytes(Q4_K, in_dim, 8))
    want, got = DevArray(nbytes=4 * n), DevArray(np.full(n, np.float32(5.0)))
    pa, pb, pc = (DevArray(np.full(nb, 0xFF, np.uint8)) for _ in range(3))
    quant.gemv_pack16_dev(xd.ptr, Q4_K, in_dim, tokens, image.ptr)
    quant.gemv_packed16_swiglu_dev(wg.ptr, wu.ptr, Q4_K, image.ptr, want.ptr, in_dim, out_dim, tokens)
    quant.gemv_pack16_dev(want.ptr, Q6_K, out_dim, tokens, pa.ptr)
    quant.gemv_packed16_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, image.ptr, got.ptr, Q6_K, pb.ptr, in_dim, out_dim, tokens)
    quant.gemv_packed16_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, image.ptr, 0, Q6_K, pc.ptr, in_dim, out_dim, tokens)
    assert np.array_equal(got.read(np.float32, n), want.read(np.float32, n))
    for p in (pb, pc):
        assert np.array_equal(p.read(np.uint8, nb), pa.read(np.uint8, nb))
    with pytest.raises(quant.QuantError, match="the next matrix is Q6_K"):
        quant.gemv_packed16_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, image.ptr, 0, Q4_K, pc.ptr, in_dim, out_dim, tokens)
    with pytest.raises(quant.QuantError, match="the next matrix is Q6_K"):
        quant.gemv_packed16_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, image.ptr, 0, Q6_K, pc.ptr, in_dim, out_dim - 16, tokens)
    for a in (wg, wu, xd, image, want, got, pa, pb, pc):
        a.close()
