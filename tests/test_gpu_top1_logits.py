"""Top-1 and logits from one pass over the weights: the ids and values of cogni_gemv_top1_dev bit for bit, and the logits that
arg-max is taken of."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K, Q8_0

pytestmark = pytest.mark.gpu


# one token and pairs on the vector ALU (walked row groups, a partial group), three and four tokens of a row only the matrix-core
# kernel takes (logits by the plain call), one pass (one and two tiles, streamed long rows, a partial tile, 11 tokens as 8 and 3)
@pytest.mark.parametrize("t,in_dim,out_dim,tokens", [(Q6_K, 4096, 32003, 1), (Q4_K, 512, 777, 2), (Q6_K, 256, 1, 1), (Q6_K, 1024, 5000, 4),
                                                     (Q4_K, 2048, 20011, 3), (Q6_K, 2048, 70001, 8), (Q4_K, 4096, 4099, 11),
                                                     (Q4_K, 12288, 530, 4), (Q6_K, 6144, 50, 6), (Q5_K, 512, 1001, 2), (Q8_0, 1024, 3584, 3)])
def test_logits_of_the_top1_pass(gpu, oracle, t, in_dim, out_dim, tokens):
    rng = np.random.default_rng(out_dim * 11 + tokens)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim)
    stride = quant.gemv_top1_partials(t, out_dim)
    print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
    wd, xd = DevArray(raw), DevArray(x)
    pi, pv = DevArray(nbytes=4 * tokens * stride), DevArray(nbytes=4 * tokens * stride)
    oi, ov, lo = DevArray(nbytes=4 * tokens), DevArray(nbytes=4 * tokens), DevArray(np.full(tokens * out_dim, np.nan, dtype=np.float32))
    want = oracle.matmul_add(x, tokens, in_dim, raw, t, out_dim, np.zeros(out_dim, dtype=np.float32), threads=8).reshape(tokens, out_dim)
    try:
        quant.gemv_top1_dev(wd.ptr, t, xd.ptr, pi.ptr, pv.ptr, oi.ptr, ov.ptr, in_dim, out_dim, tokens)
        ids, vals = oi.read(np.uint32, tokens), ov.read(np.float32, tokens)
        quant.gemv_top1_logits_dev(wd.ptr, t, xd.ptr, pi.ptr, pv.ptr, oi.ptr, ov.ptr, lo.ptr, in_dim, out_dim, tokens)
        check(oi.read(np.uint32, tokens), ov.read(np.float32, tokens), lo.read(np.float32, tokens * out_dim).reshape(tokens, out_dim), ids, vals, want)
        if t in (Q4_K, Q6_K) and tokens <= 8 and quant.gemv_image_bytes(t, in_dim, 8):
            image = DevArray(nbytes=quant.gemv_image_bytes(t, in_dim, 8))
            if tokens > 1:   # (the pack takes two tokens and more)
                quant.gemv_pack_dev(xd.ptr, t, in_dim, tokens, image.ptr)
                quant.gemv_packed_top1_dev(wd.ptr, t, image.ptr, pi.ptr, pv.ptr, oi.ptr, ov.ptr, in_dim, out_dim, tokens)
                ids, vals = oi.read(np.uint32, tokens), ov.read(np.float32, tokens)
                quant.gemv_packed_top1_logits_dev(wd.ptr, t, image.ptr, pi.ptr, pv.ptr, oi.ptr, ov.ptr, lo.ptr, in_dim, out_dim, tokens)
                check(oi.read(np.uint32, tokens), ov.read(np.float32, tokens), lo.read(np.float32, tokens * out_dim).reshape(tokens, out_dim), ids, vals, want)
            image.close()
        with pytest.raises(quant.QuantError, match="null device pointer"):
            quant.gemv_top1_logits_dev(wd.ptr, t, xd.ptr, pi.ptr, pv.ptr, oi.ptr, ov.ptr, 0, in_dim, out_dim, tokens)
    finally:
        for d in (wd, xd, pi, pv, oi, ov, lo):
            d.close()


def check(ids, vals, logits, want_ids, want_vals, want):
    assert np.array_equal(ids, want_ids) and np.array_equal(vals.view(np.uint32), want_vals.view(np.uint32))
    for m in range(len(ids)):
        assert ids[m] == int(np.argmax(logits[m])) and vals[m] == logits[m].max(), m
        # the decode kernels' bar: 22-bit activations or fp32 sums, relative to a token's largest output
        assert np.max(np.abs(logits[m].astype(np.float64) - want[m])) <= 2e-5 * np.max(np.abs(want[m])), m
