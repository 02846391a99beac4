"""The prefill kernels of 256 tokens x 256 rows: Q4_K lists, gate | up with SwiGLU."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q6_K

pytestmark = pytest.mark.gpu


def _dequantized(raw, out_dim, in_dim):
    return quant.dequantize(raw, Q4_K, out_dim * in_dim).reshape(out_dim, in_dim)


def sums_bound(oracle, raw, x, out_dim, in_dim):
    """Two fp32 sums of the same n products in different orders. x has random signs, so a partial sum stays within 6 times the products' 2-norm s; each of at
    most n roundings is off by up to 2^-24 of that, in a random direction, and n of them add up to more than 1.3 sqrt(n) of one in no output of the millions
    here: 16 sqrt(n) 2^-24 s for both sums together. (A left-out product is s / sqrt(n) on average: 85 times the bound at n = 12288, more below; the
    kernels differ by up to 5e-6 s there.)"""
    w = oracle.dequantize(raw, Q4_K, out_dim * in_dim).reshape(out_dim, in_dim)
    return 16 * np.sqrt(in_dim) * 2.0**-24 * np.sqrt(x**2 @ (w**2).T) * 1.01   # (1.01: operands rounded to half)


# token tiles that are clipped, end at a 128-token tile, are whole; matrices that end inside a tile, inside a wavefront's 64 rows, of no multiple
# of four rows, of one row; one super-block, an even and an odd number
@pytest.mark.parametrize("tokens,in_dim,dims", [(129, 256, [300]), (255, 512, [256, 1]), (256, 768, [64, 513, 7]), (257, 256, [1000, 255]),
                                                (384, 1024, [192, 256]), (513, 512, [321, 64, 100, 5, 256, 257]), (1, 256, [65])])
def test_lists(gpu, oracle, tokens, in_dim, dims):
    rng = np.random.default_rng(tokens + in_dim)
    raws = [synth.make_weights(rng, Q4_K, d, in_dim) for d in dims]
    x = synth.make_activations(rng, tokens, in_dim)
    wsb = quant.gemm_workspace_bytes(Q4_K, in_dim, tokens)
    ws, xd, wd = DevArray(nbytes=wsb), DevArray(x), [DevArray(r) for r in raws]
    outs = [[DevArray(np.full(tokens * d + 4, np.float32(-3.0))) for d in dims] for _ in range(2)]
    quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
    for w, o, d in zip(wd, outs[0], dims):
        quant.gemm_packed_dev(w.ptr, Q4_K, ws.ptr, wsb, o.ptr, in_dim, d, tokens)
    quant.gemm_tall_dev([w.ptr for w in wd], Q4_K, ws.ptr, wsb, [o.ptr for o in outs[1]], dims, in_dim, tokens)
    for raw, a, b, d in zip(raws, outs[0], outs[1], dims):
        want, got = (o.read(np.float32, tokens * d + 4) for o in (a, b))
        assert np.array_equal(got[tokens * d:], np.full(4, np.float32(-3.0)))
        diff = np.abs(want[:tokens * d].astype(np.float64) - got[:tokens * d]).reshape(tokens, d)
        assert (diff <= sums_bound(oracle, raw, x.reshape(tokens, in_dim), d, in_dim)).all(), d
    for a in [ws, xd] + wd + sum(outs, []):
        a.close()


@pytest.mark.parametrize("next_type", [Q4_K, Q6_K])
@pytest.mark.parametrize("tokens,out_dim,in_dim,keep", [(129, 256, 256, True), (256, 512, 768, True), (300, 768, 512, False), (513, 256, 1024, True)])
def test_gate_up_swiglu(gpu, tokens, out_dim, in_dim, next_type, keep):
    """Products and packed activations (absent tokens zeros) against the 128-token kernels': fp32 to 3e-6 of a token's largest product (sums in another
    order: 2-norm 6e-7, the two roundings of gemm_tall_silu 1e-7), the packed halves what those products round to."""
    rng = np.random.default_rng(tokens + next_type)
    x = synth.make_activations(rng, tokens, in_dim) * np.float32(0.05)
    wg, wu = (DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)) for _ in range(2))
    wsb, nxb = quant.gemm_workspace_bytes(Q4_K, in_dim, tokens), quant.gemm_workspace_bytes(next_type, out_dim, tokens)
    xd, ws = DevArray(x), DevArray(nbytes=wsb)
    o1, o2 = (DevArray(np.full(tokens * out_dim, np.float32(-3.0))) for _ in range(2))
    p1, p2 = (DevArray(np.full(nxb, 0xFF, np.uint8)) for _ in range(2))
    quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
    quant.gemm_packed_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, ws.ptr, wsb, o1.ptr, next_type, p1.ptr, nxb, in_dim, out_dim, tokens)
    quant.gemm_tall_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, ws.ptr, wsb, o2.ptr if keep else 0, next_type, p2.ptr, nxb, in_dim, out_dim, tokens)
    want, got = (o.read(np.float32, tokens * out_dim).reshape(tokens, out_dim) for o in (o1, o2))
    if keep:
        assert np.all(np.abs(want - got) <= 3e-6 * np.abs(want).max(axis=1, keepdims=True))
        quant.gemm_pack_dev(o2.ptr, next_type, out_dim, tokens, p1.ptr, nxb)
        assert np.array_equal(p2.read(np.uint8, nxb), p1.read(np.uint8, nxb))
    else:
        assert np.array_equal(got, np.full_like(got, -3.0))
        a, b = (p.read(np.uint8, nxb).view(np.float16).astype(np.float32) for p in (p1, p2))
        assert np.all(np.abs(a - b) <= 2.0**-10 * np.abs(a) + 3e-6 * np.abs(want).max())
    for a in (wg, wu, xd, ws, o1, o2, p1, p2):
        a.close()


@pytest.mark.parametrize("scale", [1.0, 45.0])
def test_gate_up_products_are_those_of_swiglu(gpu, scale):
    """silu(gate) * up in the epilogue against swiglu_f32 of the same sums (gemm_tall_dev adds them in the same order): one function computed two ways, each within
    an ulp of the same value at every step, so at most two ulps apart (the same bits on the MI355X); with scale 45 gates of +-200, the ones below -87.3 among
    them where 1 / (1 + e^-g) is subnormal, and gates of either infinity and NaN: the same infinities and NaNs."""
    tokens, in_dim, out_dim = 257, 512, 512
    rng = np.random.default_rng(7)
    x = synth.make_activations(rng, tokens, in_dim).reshape(tokens, in_dim)
    rg, ru = (synth.make_weights(rng, Q4_K, out_dim, in_dim) for _ in range(2))
    gates = x[:64] @ _dequantized(rg, out_dim, in_dim).T
    x *= np.float32(scale / gates.std())
    x[0], x[1], x[2, 3] = 1.0, -1.0, np.nan
    blocks = rg.reshape(out_dim, in_dim // 256, 144)
    blocks[5, :, :2], blocks[5, :, 2:4] = (0x00, 0x7C), 0   # row 5 of gate: d infinite, every scale and every code one, no minimum
    blocks[5, :, 4:8], blocks[5, :, 8:12], blocks[5, :, 12:16], blocks[5, :, 16:] = 1, 0, 1, 0x11
    n, wsb, nxb = tokens * out_dim, quant.gemm_workspace_bytes(Q4_K, in_dim, tokens), quant.gemm_workspace_bytes(Q6_K, out_dim, tokens)
    xd, ws, nx, wg, wu = DevArray(x.reshape(-1)), DevArray(nbytes=wsb), DevArray(nbytes=nxb), DevArray(rg), DevArray(ru)
    g, u, a, b = (DevArray(np.full(n, np.float32(-3.0))) for _ in range(4))
    quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
    quant.gemm_tall_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, ws.ptr, wsb, a.ptr, Q6_K, nx.ptr, nxb, in_dim, out_dim, tokens)
    quant.gemm_tall_dev([wg.ptr, wu.ptr], Q4_K, ws.ptr, wsb, [g.ptr, u.ptr], [out_dim, out_dim], in_dim, tokens)
    quant.swiglu_dev(g.ptr, u.ptr, b.ptr, n)
    gate, got, want = (v.read(np.float32, n) for v in (g, a, b))
    assert gate[5] == np.inf and gate[out_dim + 5] == -np.inf and np.isnan(gate[2 * out_dim:3 * out_dim]).all()
    if scale > 1:
        assert (gate > 150).any() and (gate < -150).any() and ((gate > -88.7) & (gate < -87.4)).sum() > 20
    assert np.array_equal(np.isnan(got), np.isnan(want)) and np.array_equal(np.isinf(got), np.isinf(want))
    finite = np.isfinite(want)
    assert np.array_equal(np.signbit(got[finite]), np.signbit(want[finite]))
    assert np.abs(got[finite].view(np.int32).astype(np.int64) - want[finite].view(np.int32)).max() <= 2
    for v in (xd, ws, nx, wg, wu, g, u, a, b):
        v.close()


@pytest.mark.parametrize("tokens,in_dim,out_dim,taken", [(998, 512, 11102, True), (1024, 512, 12287, True), (1024, 1024, 8192, False), (300, 3840, 5000, False), (643, 1280, 10773, False)])
def test_router_takes_them(gpu, tokens, in_dim, out_dim, taken):
    """cogni_matmul_dev: the bits of a pack and these tiles where the rule says so and there is no bias, else of cogni_gemm_dev."""
    rng = np.random.default_rng(tokens + out_dim)
    n, wsb = tokens * out_dim, quant.gemm_workspace_bytes(Q4_K, in_dim, tokens)
    w, x = DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)), DevArray(synth.make_activations(rng, tokens, in_dim))
    bias, ws = DevArray(synth.make_activations(rng, 1, out_dim)), DevArray(nbytes=wsb)
    a, b, c, d = (DevArray(np.full(n, np.float32(-3.0))) for _ in range(4))
    quant.matmul_dev(w.ptr, Q4_K, x.ptr, a.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
    if taken:
        quant.gemm_tall_dev([w.ptr], Q4_K, ws.ptr, wsb, [b.ptr], [out_dim], in_dim, tokens)
    else:
        quant.gemm_dev(w.ptr, Q4_K, x.ptr, b.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
    quant.matmul_dev(w.ptr, Q4_K, x.ptr, c.ptr, in_dim, out_dim, tokens, ws.ptr, wsb, bias.ptr)
    quant.gemm_dev(w.ptr, Q4_K, x.ptr, d.ptr, in_dim, out_dim, tokens, ws.ptr, wsb, bias.ptr)
    for p, q in ((a, b), (c, d)):
        assert np.array_equal(p.read(np.uint32, n), q.read(np.uint32, n))
    if taken:
        with pytest.raises(quant.QuantError, match="workspace has"):
            quant.matmul_dev(w.ptr, Q4_K, x.ptr, a.ptr, in_dim, out_dim, tokens, ws.ptr, wsb - 256)
        with pytest.raises(quant.QuantError, match="null device pointer"):
            quant.matmul_dev(w.ptr, Q4_K, 0, a.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
    for v in (w, x, bias, ws, a, b, c, d):
        v.close()


def test_which_launches_take_these_kernels(gpu):
    dims = [4096, 1024, 1024, 12288, 12288]
    assert [quant.gemm_tall_takes(Q4_K, 4096, dims, m) for m in (64, 128, 256, 384, 400, 512, 1024, 2048)] == [False] * 4 + [True] * 4
    assert not quant.gemm_tall_takes(Q6_K, 4096, dims, 512) and not quant.gemm_tall_takes(Q4_K, 4096, [4096], 512)
    assert [quant.gemm_tall_swiglu_takes(Q4_K, 4096, 12288, m) for m in (256, 512, 1024, 2048)] == [False, True, False, True]
    with pytest.raises(quant.QuantError, match="256-token tiles: Q6_K"):
        quant.gemm_tall_dev([1], Q6_K, 1, 1 << 30, [1], [256], 256, 256)
    with pytest.raises(quant.QuantError, match="workspace has"):
        quant.gemm_tall_dev([1], Q4_K, 1, 16, [1], [256], 256, 256)
