"""Two prefill matrices with an input each in one launch, both with k splits of their own (o and down of a layer)."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from cogni_ml_amd.projection_stack import QwenProjectionStackRunner, Weights
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K

pytestmark = pytest.mark.gpu


def sums_bound(oracle, raw, t, x, out_dim, in_dim):
    """Two fp32 sums of the same n products in different orders. x has random signs, so a partial sum stays within 6 times the products' 2-norm s; each of at
    most n roundings is off by up to 2^-24 of that, in a random direction, and n of them add up to more than 1.3 sqrt(n) of one in no output of the millions
    here: 16 sqrt(n) 2^-24 s for both sums together. (A left-out product is s / sqrt(n) on average: 85 times the bound at n = 12288, more below; the
    kernels differ by up to 5e-6 s there.)"""
    w = oracle.dequantize(raw, t, out_dim * in_dim).reshape(out_dim, in_dim)
    return 16 * np.sqrt(in_dim) * 2.0**-24 * np.sqrt(x**2 @ (w**2).T) * 1.01   # (1.01: operands rounded to half)


# tokens and rows that end inside a tile, inside a wavefront's rows, at them, of no multiple of four rows; no split, one matrix split, both;
# splits that do not divide the super-blocks; the fewest tokens; either order; up to the 256 tiles of a round
@pytest.mark.parametrize("tokens,a,b", [(897, (Q4_K, 512, 300), (Q6_K, 8448, 1283)), (193, (Q4_K, 2560, 2560), (Q4_K, 12288, 3072)),
                                        (1024, (Q4_K, 2048, 1024), (Q4_K, 4096, 2560)), (320, (Q6_K, 9728, 2305), (Q4_K, 2304, 2304)),
                                        (2049, (Q4_K, 256, 1), (Q6_K, 2048, 2560)), (640, (Q4_K, 2048, 1030), (Q6_K, 11008, 1536)),
                                        (300, (Q5_K, 3072, 2001), (Q6_K, 9728, 2304)), (257, (Q4_K, 10240, 2304), (Q5_K, 2304, 2304))])
def test_two_matrices(gpu, oracle, tokens, a, b):
    rng = np.random.default_rng(tokens)
    assert quant.gemm_wide_two_takes(*a, *b, tokens)
    mats, args = [], []
    for t, in_dim, out_dim in (a, b):
        raw, x = synth.make_weights(rng, t, out_dim, in_dim), synth.make_activations(rng, tokens, in_dim)
        n = quant.gemm_workspace_bytes(t, in_dim, tokens)
        w, xd, ws = DevArray(raw), DevArray(x), DevArray(nbytes=n)
        one, two = (DevArray(np.full(tokens * out_dim + 4, np.float32(-3.0))) for _ in range(2))
        quant.gemm_pack_dev(xd.ptr, t, in_dim, tokens, ws.ptr, n)
        quant.gemm_packed_dev(w.ptr, t, ws.ptr, n, one.ptr, in_dim, out_dim, tokens)
        mats.append((raw, t, x, in_dim, out_dim, w, xd, ws, one, two))
        args += [w.ptr, t, ws.ptr, n, two.ptr, in_dim, out_dim]
    size = quant.gemm_wide_two_scratch_bytes()
    scratch = DevArray(np.full(size + 64, 0xFF, np.uint8))   # (NaN in every plane that nothing writes)
    quant.gemm_wide_two_dev(*args, scratch.ptr, size, tokens)
    assert np.all(scratch.read(np.uint8, size + 64)[size:] == 0xFF)
    for raw, t, x, in_dim, out_dim, w, xd, ws, one, two in mats:
        want, got = (o.read(np.float32, tokens * out_dim + 4) for o in (one, two))
        assert np.array_equal(got[tokens * out_dim:], np.full(4, np.float32(-3.0)))
        diff = np.abs(want[:-4].astype(np.float64) - got[:-4]).reshape(tokens, out_dim)
        assert (diff <= sums_bound(oracle, raw, t, x.reshape(tokens, in_dim), out_dim, in_dim)).all(), (t, out_dim)
        for v in (w, xd, ws, one, two):
            v.close()
    scratch.close()


@pytest.mark.parametrize("down", [Q4_K, Q6_K])
def test_runner_of_the_two(gpu, down, monkeypatch):
    """The runner with and without this launch, a token count that it takes and one that it does not: the sums in another order, so fp32 to 2e-5 of a
    token's largest (11008 terms: 2-norm 4e-7)."""
    rng = np.random.default_rng(int(down))
    weights = Weights.synthetic(rng, [("q", "x", Q4_K, 2048, 2048), ("gate", "x", Q4_K, 256, 2048), ("up", "x", Q4_K, 11008, 2048),
                                      ("o", "q", Q4_K, 2048, 2048), ("down", "up", down, 2048, 11008)])
    xs = synth.make_activations(rng, 500, 2048).reshape(-1) * np.float32(0.1)
    seen, results = [], []
    f = quant.gemm_wide_two_dev
    monkeypatch.setattr(quant, "gemm_wide_two_dev", lambda *a: (seen.append(a[-2]), f(*a))[1])
    for without in (False, True):
        if without:
            monkeypatch.setattr(quant, "gemm_wide_two_takes", lambda *a: False)
        r = QwenProjectionStackRunner.from_weights(weights, 500, xs)
        r.upload_weights()
        r.reset_sequence()
        for count in (100, 500):
            r.active_tokens = count
            r.run_sequence()
        r.read_outputs()
        results.append({k: v.reshape(500, -1).copy() for k, v in r.outputs.items()})
        r.close()
    assert seen == [500]
    for k in results[0]:
        a, b = results[0][k], results[1][k]
        assert np.all(np.abs(a - b) <= 2e-5 * np.abs(b).max(axis=1, keepdims=True)), k


@pytest.mark.parametrize("tokens,in_dim,dims", [(200, 256, [16384, 8199, 5, 4100]), (65, 512, [40960, 1, 16384]), (385, 768, [7936, 8190])])
def test_q5_k_lists_of_256_row_tiles(gpu, tokens, in_dim, dims):
    """Lists that this tile takes fewer rounds for: the bits of each matrix on its own (four wavefronts, no k split)."""
    rng = np.random.default_rng(tokens)
    n = quant.gemm_workspace_bytes(Q5_K, in_dim, tokens)
    x, ws = DevArray(synth.make_activations(rng, tokens, in_dim)), DevArray(nbytes=n)
    quant.gemm_pack_dev(x.ptr, Q5_K, in_dim, tokens, ws.ptr, n)
    w = [DevArray(synth.make_weights(rng, Q5_K, d, in_dim)) for d in dims]
    one, many = ([DevArray(np.full(tokens * d + 4, np.float32(-3.0))) for d in dims] for _ in range(2))
    for a, o, d in zip(w, one, dims):
        quant.gemm_packed_dev(a.ptr, Q5_K, ws.ptr, n, o.ptr, in_dim, d, tokens)
    quant.gemm_packed_many_dev([a.ptr for a in w], Q5_K, ws.ptr, n, [o.ptr for o in many], dims, in_dim, tokens)
    for a, b, d in zip(one, many, dims):
        assert np.array_equal(a.read(np.uint32, tokens * d + 4), b.read(np.uint32, tokens * d + 4)), d
    for a in [x, ws] + w + one + many:
        a.close()


@pytest.mark.parametrize("tokens,in_dim,dims", [(9, 256, [300, 7]), (64, 512, [256, 1000]), (130, 768, [65, 513])])
def test_q5_k_lists_where_the_knob_says_so(gpu, tokens, in_dim, dims, monkeypatch):
    """COGNI_GEMM_WIDE=1: these tiles at every token count, the same bits."""
    monkeypatch.setenv("COGNI_GEMM_WIDE", "1")
    test_q5_k_lists_of_256_row_tiles(gpu, tokens, in_dim, dims)


def test_what_is_not_taken(gpu):
    takes = quant.gemm_wide_two_takes
    o, down = (Q4_K, 4096, 4096), (Q6_K, 12288, 4096)
    assert [takes(*o, *down, m) for m in (64, 192, 256, 512, 640, 1024)] == [False, False, True, True, True, False]
    assert takes(*down, *o, 512) and not takes(*down, *down, 512) and takes(Q5_K, 4096, 4096, *down, 512)
    assert not takes(Q5_K, 4096, 4096, Q5_K, 12288, 4096, 512) and not takes(Q6_K, 4096, 4096, *down, 512)
    assert not takes(Q4_K, 1792, 1792, Q6_K, 2560, 1792, 289) and not takes(Q4_K, 4096, 4096, Q6_K, 12200, 4096, 512)
    args = [64, *o[:1], 64, 1 << 30, 64, *o[1:], 64, *down[:1], 64, 1 << 30, 64, *down[1:]]
    with pytest.raises(quant.QuantError, match="not a launch for these kernels"):
        quant.gemm_wide_two_dev(*args, 64, 1 << 30, 1024)
    with pytest.raises(quant.QuantError, match="scratch too small"):
        quant.gemm_wide_two_dev(*args, 64, 1 << 20, 512)
    with pytest.raises(quant.QuantError, match="workspace has"):
        quant.gemm_wide_two_dev(*(args[:3] + [16] + args[4:]), 64, 1 << 30, 512)
