"""Several tokens of F32, F16, IQ4_NL and Q8_0 weights on the matrix cores (activations as three bfloat16 terms): fp32 precision
at every tile shape and remainder, against the oracle."""
import ctypes

import numpy as np
import pytest

from cogni_ml_amd import hip, quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import F16, F32, IQ4_NL, Q8_0

pytestmark = pytest.mark.gpu

# (in_dim, out_dim, tokens): every tile (1x1, 1x2, 2x2, 2x4, 4x4 sixteens), one more and one less than a tile, a row that ends
# inside a step of 32 (only F32 and F16 have such rows of any length; the block formats clip their last block), fewer steps than
# wavefronts, one row, one token (IQ4_NL)
CASES = [(96, 40, 9), (1024, 3584, 17), (1056, 4111, 33), (544, 2064, 64), (288, 4097, 129), (512, 4096, 200), (32, 1, 16),
         (4128, 17, 15), (1000, 33, 31), (70, 5, 65), (5, 3, 6), (2048, 300, 1), (2048, 300, 3)]


@pytest.mark.parametrize("t", [F32, F16, IQ4_NL, Q8_0])
@pytest.mark.parametrize("in_dim,out_dim,tokens", CASES)
def test_terms_kernels_match_the_oracle(gpu, oracle, t, in_dim, out_dim, tokens):
    rng = np.random.default_rng(t * 7919 + in_dim * 13 + out_dim * 7 + tokens)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim)
    x[:: 7] *= np.float32(1e-6)
    x[3:: 11] *= np.float32(1e5)                       # terms of very different size in one sum
    res = rng.standard_normal(tokens * out_dim).astype(np.float32)
    print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
    want = oracle.matmul_add(x, tokens, in_dim, raw, t, out_dim, np.zeros(out_dim, dtype=np.float32), threads=16)
    row = raw.size // out_dim
    dense = np.stack([oracle.dequantize(raw[r * row:(r + 1) * row], t, in_dim) for r in range(out_dim)]).astype(np.float64)
    mags = np.abs(x.reshape(tokens, in_dim).astype(np.float64)) @ np.abs(dense).T
    # the term product left out (fp32 weights) is below 2^-30 of a product; a sum goes through at most 32 + 2 roundings inside a
    # step of 32, one per step of a k-slice (an eighth of them), three for the slices and one for the block scale; the oracle's
    # own result is rounded once
    bound = (2.0 ** -6 + 34 + (in_dim / 32) / 8 + 1 + 3 + 1 + 1) * 2.0 ** -24 * mags.reshape(-1) + 1e-37
    w, xd, od, rd = DevArray(raw), DevArray(x), DevArray(np.full(tokens * out_dim, np.nan, dtype=np.float32)), DevArray(res)
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim)
        err = np.abs(got.astype(np.float64) - want)
        assert np.all(err <= bound), (err - bound).max()
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, rd.ptr)
        assert np.array_equal(od.read(np.float32, tokens * out_dim), got + res)
        assert quant.gemv_passes(t, tokens, in_dim, out_dim) == 1 or (t == Q8_0 and tokens <= 8)
    finally:
        for a in (w, xd, od, rd):
            a.close()


@pytest.mark.parametrize("t", [F32, F16, IQ4_NL, Q8_0])
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(96, 40, 9), (1024, 33, 33), (70, 5, 65)])
def test_infinities_and_nans_stay_what_they_are(gpu, oracle, t, in_dim, out_dim, tokens):
    """An infinity has no finite bfloat16 terms: the outputs of its row are the row kernels' (+-inf, or NaN where both signs or a
    zero weight meet), the other rows' are finite. Exactly: which outputs are finite, +inf, -inf and NaN."""
    rng = np.random.default_rng(t * 31 + in_dim + tokens)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim).reshape(tokens, in_dim)
    x[0, 3] = np.inf
    x[2, in_dim - 1] = -np.inf
    x[4, 0], x[4, in_dim // 2] = np.inf, -np.inf
    x[5, 1] = np.nan
    x[6, 2] = np.uint32(0x7F800001).view(np.float32)   # a NaN whose upper half is that of an infinity
    want = oracle.matmul_add(x, tokens, in_dim, raw, t, out_dim, np.zeros(out_dim, dtype=np.float32), threads=4).reshape(tokens, out_dim)
    w, xd, od = DevArray(raw), DevArray(x), DevArray(np.zeros(tokens * out_dim, dtype=np.float32))
    try:
        print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
    finally:
        for a in (w, xd, od):
            a.close()
    for kind in (np.isfinite, np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(got), kind(want)), kind.__name__


@pytest.mark.parametrize("t", [F32, F16])
@pytest.mark.parametrize("in_dim", [1, 2, 3])
def test_no_term_product_is_missing(gpu, t, in_dim):
    """Values whose bfloat16 terms behind the first are as large as they get, all of one sign: a term product left out shows (the
    smallest of them is 3.3 * 2^-24 of the sum with binary16 weights, as much each with fp32). Bound: a matrix instruction may drop
    what lies below the last place of its result (2 * 2^-24, here that of the sum of the smaller term products as the leading one
    joins it; 2^-6 of that before), and one rounding of the result."""
    out_dim, tokens = 20, 6
    rng = np.random.default_rng(in_dim + t)
    x = (np.full((tokens, in_dim), 0x3F80FFFF, dtype=np.uint32).view(np.float32) * np.float32(2.0) ** rng.integers(-3, 4, (tokens, 1))).astype(np.float32)
    if t == F32:
        dense = (np.full((out_dim, in_dim), 0x3F80FFFF, dtype=np.uint32).view(np.float32) * np.float32(2.0) ** rng.integers(-3, 4, (out_dim, 1))).astype(np.float32)
    else:
        dense = (np.full((out_dim, in_dim), 0x3C07, dtype=np.uint16).view(np.float16) * np.float16(2.0) ** rng.integers(-3, 4, (out_dim, 1))).astype(np.float16)
    want = x.astype(np.float64) @ dense.astype(np.float64).T
    w, xd, od = DevArray(dense), DevArray(x), DevArray(np.full(tokens * out_dim, np.nan, dtype=np.float32))
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
    finally:
        for a in (w, xd, od):
            a.close()
    err = np.abs(got.astype(np.float64) - want) / want * 2.0 ** 24
    assert err.max() <= 3 + 2.0 ** -4, err.max()


@pytest.mark.parametrize("t,kernel", [(F32, "f32_gemv_plain_f32"), (F16, "f16_gemv_plain_f32"), (IQ4_NL, "iq4_nl_gemv_plain_f32")])
@pytest.mark.parametrize("in_dim", [256, 1024, 4096])
@pytest.mark.parametrize("positive", [False, True])
def test_no_further_from_64_bits_than_the_row_kernel(gpu, oracle, t, kernel, in_dim, positive):
    """The error in the 2-norm against 64-bit sums of the row kernel (a chain of fused multiply-adds per lane) on the same inputs, of
    mixed signs and all of one: not exceeded but by what another order of the same number of roundings changes (a tenth)."""
    out_dim, tokens = 512, 33
    rng = np.random.default_rng(t + in_dim + positive)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim).reshape(tokens, in_dim)
    if positive:
        x = np.abs(x)
        if t == F32:
            raw = np.abs(raw.view(np.float32)).view(np.uint8)
        elif t == F16:
            raw = np.abs(raw.view(np.float16)).view(np.uint8)
        else:
            raw.reshape(-1, 18)[:, 2:] |= 0x88   # the upper half of the table is positive
    row = raw.size // out_dim
    dense = np.stack([oracle.dequantize(raw[r * row:(r + 1) * row], t, in_dim) for r in range(out_dim)]).astype(np.float64)
    want = x.astype(np.float64) @ dense.T
    w, xd, od = DevArray(raw), DevArray(x), DevArray(nbytes=4 * tokens * out_dim)
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
        params = hip.KernelParams(*[ctypes.c_uint64(v) for v in (w.ptr, xd.ptr, 0, od.ptr)], *[ctypes.c_uint32(v) for v in (in_dim, out_dim, tokens)])
        module = hip.HIPModule.load_builtin()
        hip.launch(module.function(kernel), (out_dim + 3) // 4, 1, 1, 256, 1, 1, params, kernel)
        rows = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
        module.close()
    finally:
        for a in (w, xd, od):
            a.close()
    assert np.linalg.norm(rows - want) <= 1e-6 * np.linalg.norm(want)
    assert np.linalg.norm(got - want) <= 1.1 * np.linalg.norm(rows - want)


@pytest.mark.parametrize("t", [Q8_0, IQ4_NL])
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(1024, 33, 9), (288, 100, 70)])
def test_activations_near_the_top_of_the_fp32_range(gpu, oracle, t, in_dim, out_dim, tokens):
    """|x| of 1e35 and more, outputs up to 1e38: a block's codes times x leave the fp32 range before the scale brings them back, the
    result does not. It is finite in the oracle's 64-bit sums and has to be here, to the bar of the one-pass kernels."""
    rng = np.random.default_rng(t + in_dim)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim).reshape(tokens, in_dim)
    x[0] *= np.float32(1e35)
    x[1] *= np.float32(1e36)
    x[tokens - 1, in_dim - 32:] *= np.float32(2e36)
    want = oracle.matmul_add(x, tokens, in_dim, raw, t, out_dim, np.zeros(out_dim, dtype=np.float32), threads=4).reshape(tokens, out_dim)
    assert np.isfinite(want).all()
    w, xd, od = DevArray(raw), DevArray(x), DevArray(nbytes=4 * tokens * out_dim)
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
    finally:
        for a in (w, xd, od):
            a.close()
    assert np.isfinite(got).all()
    for m in range(tokens):
        assert np.max(np.abs(got[m].astype(np.float64) - want[m])) <= 2e-5 * np.max(np.abs(want[m]).astype(np.float64)), m


@pytest.mark.parametrize("t", [F32, F16])
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(96, 40, 9), (1024, 70, 33), (512, 4097, 129), (70, 5, 65)])
def test_infinite_weights_leave_the_other_rows_alone(gpu, oracle, t, in_dim, out_dim, tokens):
    """Rows with an infinity, two of both signs and a NaN, in the first and in the last (partial) tile: which outputs are finite,
    +inf, -inf and NaN is what the oracle says, with and without a residual, and every other output keeps its bits."""
    rng = np.random.default_rng(t + in_dim + out_dim)
    dense = synth.make_weights(rng, t, out_dim, in_dim).view(np.float32 if t == F32 else np.float16).reshape(out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim).reshape(tokens, in_dim)
    x[1, 0] = 0.0
    res = rng.standard_normal(tokens * out_dim).astype(np.float32)
    bad = dense.copy()
    bad[0, 0] = np.inf                      # NaN against the zero of token 1
    bad[2, 3], bad[2, in_dim - 1] = np.inf, -np.inf
    bad[out_dim - 1, in_dim // 2] = -np.inf
    bad[out_dim - 2, in_dim - 1] = np.nan
    touched = [0, 2, out_dim - 1, out_dim - 2]
    want = oracle.matmul_add(x, tokens, in_dim, np.ascontiguousarray(bad[touched]).view(np.uint8).reshape(-1), t, 4, np.zeros(4, dtype=np.float32),
                             threads=4).reshape(tokens, 4)
    good, w, xd, rd, od = DevArray(dense), DevArray(bad), DevArray(x), DevArray(res), DevArray(nbytes=4 * tokens * out_dim)
    try:
        print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
        quant.gemv_dev(good.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        plain = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
        quant.gemv_dev(w.ptr, t, xd.ptr, rd.ptr, in_dim, out_dim, tokens, rd.ptr)   # in place
        added = rd.read(np.float32, tokens * out_dim).reshape(tokens, out_dim)
    finally:
        for a in (good, w, xd, rd, od):
            a.close()
    rest = np.setdiff1d(np.arange(out_dim), touched)
    assert np.array_equal(got[:, rest], plain[:, rest])
    assert np.array_equal(added[:, rest], plain[:, rest] + res.reshape(tokens, out_dim)[:, rest])
    for kind in (np.isfinite, np.isposinf, np.isneginf, np.isnan):
        assert np.array_equal(kind(got[:, touched]), kind(want)), kind.__name__
        assert np.array_equal(kind(added[:, touched]), kind(want)), kind.__name__


@pytest.mark.parametrize("t", [F32, F16, Q8_0, IQ4_NL])
@pytest.mark.parametrize("x_exp,w_exp", [(-112, 0), (-120, 10), (-128, 10), (-140, 15), (60, -130)])
def test_activations_near_the_bottom_of_the_fp32_range(gpu, oracle, t, x_exp, w_exp):
    """Values whose bfloat16 terms, some or all, are below the smallest normal one (the values themselves below it, too), against
    weights of any size: the error bound of every other input, and half a last place where the result is subnormal."""
    in_dim, out_dim, tokens = 544, 70, 33
    if t != F32 and w_exp < 0:
        pytest.skip("binary16 weights and block scales do not reach that far down")
    rng = np.random.default_rng(t + 1000 - x_exp)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    if t == F32:
        raw = (raw.view(np.float32) * np.float32(2.0) ** w_exp).astype(np.float32).view(np.uint8)
    elif t == F16:
        raw = (raw.view(np.float16) * np.float16(2.0) ** min(w_exp, 10)).astype(np.float16).view(np.uint8)
    x = (synth.make_activations(rng, tokens, in_dim).astype(np.float64) * 2.0 ** x_exp).astype(np.float32).reshape(tokens, in_dim)
    row = raw.size // out_dim
    dense = np.stack([oracle.dequantize(raw[r * row:(r + 1) * row], t, in_dim) for r in range(out_dim)]).astype(np.float64)
    want, mags = x.astype(np.float64) @ dense.T, np.abs(x.astype(np.float64)) @ np.abs(dense).T
    # as in test_terms_kernels_match_the_oracle (17 steps of 32)
    bound = (2.0 ** -6 + 34 + 17 / 8 + 1 + 3 + 1) * 2.0 ** -24 * mags + 2.0 ** -150
    w, xd, od = DevArray(raw), DevArray(x), DevArray(nbytes=4 * tokens * out_dim)
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        got = od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim).astype(np.float64)
    finally:
        for a in (w, xd, od):
            a.close()
    assert np.all(np.abs(got - want) <= bound), (np.abs(got - want) / mags).max()
    assert np.linalg.norm(got - want) <= 2.0 ** -22 * np.linalg.norm(want) + 2.0 ** -150 * np.sqrt(want.size)


@pytest.mark.parametrize("t", [F32, F16])
def test_more_tokens_than_a_launch_has_threads_for(gpu, t):
    """2^24 tokens of one tile of rows are 2^23 workgroups of 512 threads, and a launch has fewer than 2^32: the call goes in several.
    The weights are powers of two and zeros, so every output is exact."""
    in_dim, out_dim, tokens = 3, 2, (1 << 24) + 17
    dense = np.array([[0, 0, -0.5], [2, 0, 0]], dtype=np.float32 if t == F32 else np.float16)
    x = np.random.default_rng(t).standard_normal((tokens, in_dim), dtype=np.float32)
    want = np.stack([x[:, 2] * np.float32(-0.5), x[:, 0] * np.float32(2)], axis=1)
    w, xd, od = DevArray(dense), DevArray(x), DevArray(np.full((tokens, out_dim), np.nan, dtype=np.float32))
    try:
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens)
        assert np.array_equal(od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim), want)
        quant.gemv_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, od.ptr)   # in place
        assert np.array_equal(od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim), want + want)
        assert quant.gemv_passes(t, tokens, in_dim, out_dim) == 2 and quant.gemv_passes(t, 1 << 20, in_dim, out_dim) == 1
    finally:
        for a in (w, xd, od):
            a.close()


@pytest.mark.parametrize("t,prefix,tm,tn,name", [(IQ4_NL, "iq4_nl", 2, 4, "2x4"), (F32, "f32", 2, 2, "2x2"), (F16, "f16", 2, 2, "2x2"), (IQ4_NL, "iq4_nl", 2, 2, "2x2"),
                                                 (Q8_0, "q8_0", 2, 2, "2x2"), (F16, "f16", 2, 4, "2x4"), (Q8_0, "q8_0", 2, 4, "2x4")])
@pytest.mark.parametrize("in_dim", [32, 70, 300, 544, 4096])
def test_both_orders_of_a_step_give_the_same_bits(gpu, t, prefix, tm, tn, name, in_dim):
    """The interleaved kernel of a tile and the other, launched by name: one step, fewer than wavefronts, a row that ends inside one, many; tiles that end
    behind the last row and token, one row of tiles for each XCD."""
    out_dim, tokens = 16 * tn * 8 - 3, 16 * tm * 3 - 5
    rng = np.random.default_rng(t + in_dim)
    w, x = DevArray(synth.make_weights(rng, t, out_dim, in_dim)), DevArray(synth.make_activations(rng, tokens, in_dim))
    res = DevArray(synth.make_activations(rng, tokens, out_dim))
    outs = [DevArray(np.full(tokens * out_dim + 4, np.float32(-3.0))) for _ in range(2)]
    module = hip.HIPModule.load_builtin()
    try:
        for o, suffix in zip(outs, ("", "_i")):
            kernel = "%s_gemm_terms_f32_%s%s" % (prefix, name, suffix)
            params = hip.KernelParams(*[ctypes.c_uint64(v) for v in (w.ptr, x.ptr, res.ptr, o.ptr)], *[ctypes.c_uint32(v) for v in (in_dim, out_dim, tokens)])
            hip.launch(module.function(kernel), 3 * 8, 1, 1, 512, 1, 1, params, kernel)
        a, b = (o.read(np.uint32, tokens * out_dim + 4) for o in outs)
        assert np.array_equal(a, b) and np.all(a[tokens * out_dim:].view(np.float32) == -3.0)
    finally:
        module.close()
        for v in [w, x, res] + outs:
            v.close()


@pytest.mark.parametrize("t,out_dim,tokens,in_dim", [(F32, 3584, 47, 1184), (F16, 2049, 60, 1540), (IQ4_NL, 3001, 35, 1408), (Q8_0, 924, 227, 1152),
                                                     (F16, 1796, 189, 1536), (IQ4_NL, 1605, 173, 2560), (Q8_0, 1605, 173, 1696)])
def test_rows_long_enough_for_the_interleaved_kernels(gpu, oracle, t, out_dim, tokens, in_dim):
    """gemv_dev where it takes them, to the bound of test_terms_kernels_match_the_oracle."""
    test_terms_kernels_match_the_oracle(gpu, oracle, t, in_dim, out_dim, tokens)


def test_token_limit_of_a_launch(gpu):
    """The launches of one call, by the number of rows; matrices of 2^27 rows keep the kernels that walk them."""
    for out_dim in (1, 129, 3584, 151936, 1 << 26):
        tiles = -(-out_dim // 128) * 8
        most = ((1 << 32) - 1) // 512 // tiles * 16
        assert quant.gemv_passes(IQ4_NL, most, 32, out_dim) == 1 and quant.gemv_passes(IQ4_NL, most + 1, 32, out_dim) == 2
    assert quant.gemv_passes(IQ4_NL, 100, 32, (1 << 27) + 1) == 1
