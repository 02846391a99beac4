"""The short-prefill GEMM kernels (weights streamed, four k-slices per workgroup) against the oracle and the tile kernels."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K

pytestmark = pytest.mark.gpu

# (in_dim, out_dim, tokens): one super-block (three of the four k-slices idle), five (uneven slices), a k split; one row, rows that
# end inside a tile and inside a group of four, tall enough for 64-row tiles; one more and one less than a token tile, the
# last token tile empty but for one
CASES = [(256, 32, 18), (256, 1, 32), (1280, 33, 33), (1024, 100, 64), (512, 8200, 31), (768, 6147, 65), (12288, 70, 48),
         (4096, 64, 129), (2048, 130, 97)]


def order_bound(oracle, raw, t, x16, in_dim, out_dim):
    """What another order of the additions may change of a sum, per element: the products of binary16 values are exact in fp32, a
    matrix instruction adds sixteen of them in at most two roundings, and a rounding is at most 2^-24 of the partial sum, which is
    on average below four times the 2-norm of the products (they have random signs). The tile kernel walks the whole row, a k-slice
    of the others a quarter of it."""
    dense = oracle.dequantize(raw, t, out_dim * in_dim).reshape(out_dim, in_dim).astype(np.float16).astype(np.float64)
    products = np.sqrt((x16.astype(np.float64) ** 2) @ (dense ** 2).T)
    return (2 * (in_dim / 16) * 1.25 + 16) * 2.0 ** -24 * 4 * products


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("in_dim,out_dim,tokens", CASES)
def test_router_and_residual(gpu, oracle, t, in_dim, out_dim, tokens):
    """The router takes these shapes to the new kernels: within the GEMM's bound of the oracle, a bias and a residual on top of
    the very same sums, and the sums those of the tile kernel up to the order of fp32 additions."""
    assert quant.gemm_stream_takes(t, in_dim, out_dim, tokens)
    rng = np.random.default_rng(t * 7919 + in_dim * 13 + out_dim * 7 + tokens)
    raw = synth.make_weights(rng, t, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim)
    bias, res = rng.standard_normal(out_dim).astype(np.float32), rng.standard_normal(tokens * out_dim).astype(np.float32)
    print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
    wsb = quant.gemm_workspace_bytes(t, in_dim, tokens, out_dim)
    w, xd, ws = DevArray(raw), DevArray(x), DevArray(nbytes=wsb)
    od, rd, bd = DevArray(np.full(tokens * out_dim + 64, np.nan, dtype=np.float32)), DevArray(res), DevArray(bias)
    try:
        quant.matmul_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
        got = od.read(np.float32, tokens * out_dim + 64)
        assert np.isnan(got[tokens * out_dim:]).all()          # nothing behind the output
        got = got[:tokens * out_dim]
        rows = rng.choice(tokens, min(tokens, 8), replace=False)
        want = oracle.matmul_add(np.ascontiguousarray(x.reshape(tokens, in_dim)[rows]).reshape(-1), len(rows), in_dim, raw, t, out_dim,
                                 np.zeros(out_dim, dtype=np.float32), threads=16).reshape(len(rows), out_dim)
        # binary16 activations and weights: the bound of every GEMM here
        assert np.abs(got.reshape(tokens, out_dim)[rows].astype(np.float64) - want).max() <= 2e-3 * np.abs(want).max()
        quant.gemm_packed_dev(w.ptr, t, ws.ptr, wsb, od.ptr, in_dim, out_dim, tokens)
        tile = od.read(np.float32, tokens * out_dim)
        bound = order_bound(oracle, raw, t, x.reshape(tokens, in_dim).astype(np.float16), in_dim, out_dim)
        worst = (np.abs(got.astype(np.float64) - tile).reshape(tokens, out_dim) / bound).max()
        print("difference from the tile kernel: %.3f of its bound" % worst, flush=True)
        assert worst <= 1
        assert np.linalg.norm(got - tile) <= 1e-5 * np.linalg.norm(tile)
        quant.matmul_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, ws.ptr, wsb, bd.ptr)
        assert np.array_equal(od.read(np.float32, tokens * out_dim).reshape(tokens, out_dim), got.reshape(tokens, out_dim) + bias)
        quant.gemm_stream_dev([w.ptr], t, ws.ptr, wsb, [rd.ptr], [out_dim], in_dim, tokens, rd.ptr)   # in place
        assert np.array_equal(rd.read(np.float32, tokens * out_dim), got + res)
    finally:
        for a in (w, xd, ws, od, rd, bd):
            a.close()


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("in_dim,out_dim", [(256, 32), (2048, 520), (4096, 1030)])
def test_seventeen_tokens(gpu, oracle, t, in_dim, out_dim):
    """The runners' launches start here, the router's one token later: at seventeen it gives the bits of cogni_gemm_dev, and the
    new kernels the same sums in another order."""
    tokens = 17
    assert quant.gemm_stream_takes(t, in_dim, out_dim, tokens) and not quant.gemm_stream_takes(t, in_dim, out_dim, 16)
    rng = np.random.default_rng(t + in_dim + out_dim)
    raw, x = synth.make_weights(rng, t, out_dim, in_dim), synth.make_activations(rng, tokens, in_dim)
    n, wsb = tokens * out_dim, quant.gemm_workspace_bytes(t, in_dim, tokens, out_dim)
    w, xd, ws, od = DevArray(raw), DevArray(x), DevArray(nbytes=wsb), DevArray(np.full(n + 64, np.nan, dtype=np.float32))
    try:
        print("case type=%d in_dim=%d out_dim=%d tokens=%d" % (t, in_dim, out_dim, tokens), flush=True)
        quant.gemm_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
        tile = od.read(np.float32, n)
        quant.matmul_dev(w.ptr, t, xd.ptr, od.ptr, in_dim, out_dim, tokens, ws.ptr, wsb)
        assert np.array_equal(od.read(np.float32, n), tile)
        quant.gemm_pack_dev(xd.ptr, t, in_dim, tokens, ws.ptr, wsb)
        quant.gemm_stream_dev([w.ptr], t, ws.ptr, wsb, [od.ptr], [out_dim], in_dim, tokens)
        got = od.read(np.float32, n + 64)
        assert np.isnan(got[n:]).all()
        bound = order_bound(oracle, raw, t, x.reshape(tokens, in_dim).astype(np.float16), in_dim, out_dim)
        assert np.all(np.abs(got[:n].astype(np.float64) - tile).reshape(tokens, out_dim) <= bound)
    finally:
        for a in (w, xd, ws, od):
            a.close()


@pytest.mark.parametrize("t", [Q4_K, Q5_K, Q6_K])
@pytest.mark.parametrize("tokens", [24, 70])
def test_list_of_matrices(gpu, t, tokens):
    """Every output of a list is that of the matrix by itself, unsplit, up to the tile height (which does not enter the sums)."""
    in_dim, outs = 1536, [512, 33, 1, 260, 64]
    rng = np.random.default_rng(tokens + t)
    raws = [DevArray(synth.make_weights(rng, t, o, in_dim)) for o in outs]
    xd = DevArray(synth.make_activations(rng, tokens, in_dim))
    wsb = quant.gemm_workspace_bytes(t, in_dim, tokens)
    ws = DevArray(nbytes=wsb)
    ods = [DevArray(np.full(tokens * o, np.nan, dtype=np.float32)) for o in outs]
    try:
        quant.gemm_pack_dev(xd.ptr, t, in_dim, tokens, ws.ptr, wsb)
        quant.gemm_stream_dev([w.ptr for w in raws], t, ws.ptr, wsb, [o.ptr for o in ods], outs, in_dim, tokens)
        got = [o.read(np.float32, tokens * n) for o, n in zip(ods, outs)]
        for w, o, n, g in zip(raws, ods, outs, got):
            quant.gemm_stream_dev([w.ptr], t, ws.ptr, wsb, [o.ptr], [n], in_dim, tokens)
            assert np.array_equal(o.read(np.float32, tokens * n), g)
    finally:
        for a in raws + ods + [xd, ws]:
            a.close()


@pytest.mark.parametrize("next_type", [Q4_K, Q6_K])
@pytest.mark.parametrize("in_dim,out_dim,tokens", [(256, 256, 17), (1280, 768, 33), (4096, 512, 64), (512, 256, 130), (256, 256, 70)])
def test_gate_up_swiglu_pack(gpu, in_dim, out_dim, tokens, next_type):
    """silu(gate) * up within a few roundings of the tile kernel's, and the packed block what the pack kernel makes of it: the
    absent tokens of the last tile of a workgroup (32 tokens up to 32, else 64) are zeros, nothing else is written."""
    rng = np.random.default_rng(in_dim + out_dim + tokens)
    g, u = (DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)) for _ in range(2))
    xd = DevArray(synth.make_activations(rng, tokens, in_dim))
    wsb, nxb = quant.gemm_workspace_bytes(Q4_K, in_dim, tokens), quant.gemm_workspace_bytes(next_type, out_dim, tokens)
    ones = np.full(nxb + 256, 0xFF, dtype=np.uint8)
    ws, nx, nx2, ref, out = DevArray(nbytes=wsb), DevArray(ones), DevArray(ones), DevArray(nbytes=nxb), DevArray(nbytes=4 * tokens * out_dim)
    try:
        quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
        quant.gemm_packed_swiglu_dev(g.ptr, u.ptr, Q4_K, ws.ptr, wsb, out.ptr, in_dim, out_dim, tokens)
        tile = out.read(np.float32, tokens * out_dim)
        quant.gemm_stream_swiglu_pack_dev(g.ptr, u.ptr, Q4_K, ws.ptr, wsb, out.ptr, next_type, nx.ptr, nxb, in_dim, out_dim, tokens)
        got, packed = out.read(np.float32, tokens * out_dim), nx.read(np.uint8, nxb + 256)
        assert np.linalg.norm(got - tile) <= 2e-5 * np.linalg.norm(tile)
        assert (packed[nxb:] == 0xFF).all()
        quant.gemm_pack_dev(out.ptr, next_type, out_dim, tokens, ref.ptr, nxb)

        def by_token(b):   # a packed block is [128 tokens][super-block][32 cells][token][16 bytes]
            return b.reshape(-1, out_dim // 256, 32, 128, 16).transpose(0, 3, 1, 2, 4).reshape(-1, out_dim // 256 * 512)
        mine, want = by_token(packed[:nxb]), by_token(ref.read(np.uint8, nxb))
        tile_tokens = 32 if tokens <= 32 else 64
        end = -(-tokens // tile_tokens) * tile_tokens
        assert np.array_equal(mine[:tokens], want[:tokens])
        assert (mine[tokens:end] == 0).all() and (mine[end:] == 0xFF).all()
        quant.gemm_stream_swiglu_pack_dev(g.ptr, u.ptr, Q4_K, ws.ptr, wsb, 0, next_type, nx2.ptr, nxb, in_dim, out_dim, tokens)
        assert np.array_equal(nx2.read(np.uint8, nxb + 256), packed)
    finally:
        for a in (g, u, xd, ws, nx, nx2, ref, out):
            a.close()


# both orders, both token tiles, with and without k splits, uneven rows; a pair that takes 64 rows and a pair without the kernel go one by one
@pytest.mark.parametrize("tokens", [18, 48, 70])
@pytest.mark.parametrize("a,b", [((Q4_K, 4096, 4096), (Q6_K, 12288, 4096)), ((Q6_K, 3072, 1030), (Q5_K, 1024, 130)), ((Q4_K, 256, 1), (Q4_K, 2816, 33)),
                                 ((Q5_K, 512, 4096), (Q4_K, 1280, 515)), ((Q4_K, 1024, 12288), (Q6_K, 256, 70)), ((Q6_K, 512, 40), (Q6_K, 256, 33))])
def test_two_matrices_with_an_input_each(gpu, a, b, tokens):
    """The launch of two matrices: each output as cogni_gemm_stream_dev gives it, bit for bit."""
    rng = np.random.default_rng(a[1] + b[1] + tokens)
    mats = []
    for t, in_dim, out_dim in (a, b):
        x, nb = DevArray(synth.make_activations(rng, tokens, in_dim)), quant.gemm_workspace_bytes(t, in_dim, tokens, out_dim)
        ws, w = DevArray(nbytes=nb), DevArray(synth.make_weights(rng, t, out_dim, in_dim))
        one, two = (DevArray(np.full(tokens * out_dim + 64, np.float32(v))) for v in (5.0, 6.0))
        quant.gemm_pack_dev(x.ptr, t, in_dim, tokens, ws.ptr, nb)
        quant.gemm_stream_dev([w.ptr], t, ws.ptr, nb, [one.ptr], [out_dim], in_dim, tokens)
        mats.append((w, t, ws, nb, two, in_dim, out_dim, one, x))
    print("case", a, b, tokens, flush=True)
    args = [v for w, t, ws, nb, two, in_dim, out_dim, one, x in mats for v in (w.ptr, t, ws.ptr, nb, two.ptr, in_dim, out_dim)]
    quant.gemm_stream_two_dev(*args, tokens)
    for w, t, ws, nb, two, in_dim, out_dim, one, x in mats:
        got = two.read(np.float32, tokens * out_dim + 64)
        assert np.array_equal(got[:tokens * out_dim], one.read(np.float32, tokens * out_dim)), (t, in_dim, out_dim)
        assert (got[tokens * out_dim:] == 6.0).all()
    with pytest.raises(quant.QuantError, match="null device pointer"):
        quant.gemm_stream_two_dev(*args[:4], 0, *args[5:], tokens)
    for m in mats:
        for i in (0, 2, 4, 7, 8):
            m[i].close()


@pytest.mark.parametrize("a,b", [((Q4_K, 96), (Q5_K, 1024)), ((Q5_K, 1024), (Q4_K, 1024))])
def test_two_matrices_of_one_workspace(gpu, a, b):
    """Both read the same packed activations and put the planes of their k splits behind them: each output as alone, bit for bit."""
    in_dim, tokens = 12288, 48   # (rows long enough for a k split)
    rng = np.random.default_rng(a[1] + b[1])
    x, nb = DevArray(synth.make_activations(rng, tokens, in_dim)), max(quant.gemm_workspace_bytes(t, in_dim, tokens, d) for t, d in (a, b))
    assert nb >= quant.gemm_workspace_bytes(Q4_K, in_dim, tokens) + 2 * 4 * tokens * max(a[1], b[1])   # room for planes
    ws = DevArray(nbytes=nb)
    quant.gemm_pack_dev(x.ptr, Q4_K, in_dim, tokens, ws.ptr, nb)
    mats = []
    for t, d in (a, b):
        w, one, two = DevArray(synth.make_weights(rng, t, d, in_dim)), DevArray(nbytes=4 * tokens * d), DevArray(nbytes=4 * tokens * d)
        quant.gemm_stream_dev([w.ptr], t, ws.ptr, nb, [one.ptr], [d], in_dim, tokens)
        mats.append((w, t, two, d, one))
    quant.gemm_stream_two_dev(*[v for w, t, two, d, one in mats for v in (w.ptr, t, ws.ptr, nb, two.ptr, in_dim, d)], tokens)
    for w, t, two, d, one in mats:
        assert np.array_equal(two.read(np.float32, tokens * d), one.read(np.float32, tokens * d)), (t, d)
        for dev in (w, two, one):
            dev.close()
    x.close()
    ws.close()
