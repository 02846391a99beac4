"""The eight-wavefront prefill kernels (128 tokens x 256 rows): lists and gate | up with SwiGLU for Q4_K, single matrices for Q6_K.
Same operands, the same k halves added in the same order as in the four-wavefront kernels: bit for bit their values."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu, launched_blocks  # noqa: F401
from helpers import Q4_K, Q6_K
from test_gpu_gemm import check, run_gemm

pytestmark = pytest.mark.gpu


# the first three: 192-row tiles in one round of 256 workgroups. The others: two rounds of those and of the 128-row ones, one of 256-row
# tiles; whole and clipped tiles, a row count that is no multiple of four, matrices that end inside a tile, super-blocks odd and even
@pytest.mark.parametrize("tokens,in_dim,dims,block", [
    (130, 256, [16001, 4101, 1000], 256), (255, 768, [8192, 8192 + 37], 256), (257, 512, [300, 7, 14000], 256),
    (255, 256, [24001, 4101, 1000], 512), (130, 768, [16384, 8192 + 37, 300], 512), (257, 512, [300, 7, 20000], 512)])
def test_lists(gpu, tokens, in_dim, dims, block, monkeypatch):
    rng = np.random.default_rng(tokens)
    raws = [synth.make_weights(rng, Q4_K, d, in_dim) for d in dims]
    x = synth.make_activations(rng, tokens, in_dim)
    wsb = quant.gemm_workspace_bytes(Q4_K, in_dim, tokens)
    ws, xd, wd = DevArray(nbytes=wsb), DevArray(x), [DevArray(r) for r in raws]
    outs = [[DevArray(np.full(tokens * d, np.float32(-3.0))) for d in dims] for _ in range(4)]
    quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
    monkeypatch.setenv("COGNI_GEMM_WIDE", "0")
    for w, o, d in zip(wd, outs[0], dims):
        quant.gemm_packed_dev(w.ptr, Q4_K, ws.ptr, wsb, o.ptr, in_dim, d, tokens)
    want = [o.read(np.float32, tokens * d) for o, d in zip(outs[0], dims)]
    for knob, expect, out in (("0", 256, outs[1]), ("1", 512, outs[2]), (None, block, outs[3])):
        if knob is None:
            monkeypatch.delenv("COGNI_GEMM_WIDE")
        else:
            monkeypatch.setenv("COGNI_GEMM_WIDE", knob)

        def issue(stream=None):
            quant.gemm_packed_many_dev([w.ptr for w in wd], Q4_K, ws.ptr, wsb, [o.ptr for o in out], dims, in_dim, tokens, stream)
        assert launched_blocks(issue) == [expect], knob
        issue()
        for o, a, d in zip(out, want, dims):
            assert np.array_equal(o.read(np.float32, tokens * d), a), (knob, d)
    for a in [ws, xd] + wd + sum(outs, []):
        a.close()


@pytest.mark.parametrize("next_type", [Q4_K, Q6_K])
@pytest.mark.parametrize("tokens,out_dim,in_dim", [(130, 13056, 256), (255, 16384, 512), (385, 6400, 768)])
def test_gate_up_swiglu(gpu, tokens, out_dim, in_dim, next_type, monkeypatch):
    """Against the two GEMMs on the four-wavefront kernels, swiglu_f32 and the pack launch: products and packed activations."""
    rng = np.random.default_rng(tokens + next_type)
    x = synth.make_activations(rng, tokens, in_dim)
    wg, wu = (DevArray(synth.make_weights(rng, Q4_K, out_dim, in_dim)) for _ in range(2))
    wsb, nxb = quant.gemm_workspace_bytes(Q4_K, in_dim, tokens), quant.gemm_workspace_bytes(next_type, out_dim, tokens)
    xd, ws = DevArray(x), DevArray(nbytes=wsb)
    g, u, o1, o2, o3 = (DevArray(np.full(tokens * out_dim, np.float32(-3.0))) for _ in range(5))
    p1, p2 = (DevArray(np.full(nxb, 0xFF, np.uint8)) for _ in range(2))
    quant.gemm_pack_dev(xd.ptr, Q4_K, in_dim, tokens, ws.ptr, wsb)
    monkeypatch.setenv("COGNI_GEMM_WIDE", "0")
    for w, o in ((wg, g), (wu, u)):
        quant.gemm_packed_dev(w.ptr, Q4_K, ws.ptr, wsb, o.ptr, in_dim, out_dim, tokens)
    quant.swiglu_dev(g.ptr, u.ptr, o1.ptr, tokens * out_dim)
    quant.gemm_pack_dev(o1.ptr, next_type, out_dim, tokens, p1.ptr, nxb)

    def issue(stream=None):
        quant.gemm_packed_swiglu_dev(wg.ptr, wu.ptr, Q4_K, ws.ptr, wsb, o2.ptr, in_dim, out_dim, tokens, stream)
        quant.gemm_packed_swiglu_pack_dev(wg.ptr, wu.ptr, Q4_K, ws.ptr, wsb, o3.ptr, next_type, p2.ptr, nxb, in_dim, out_dim, tokens, stream)
    assert launched_blocks(issue) == [256, 256]
    monkeypatch.delenv("COGNI_GEMM_WIDE")
    assert launched_blocks(issue) == [512, 512]
    issue()
    want = o1.read(np.float32, tokens * out_dim)
    assert np.array_equal(o2.read(np.float32, want.size), want)
    assert np.array_equal(o3.read(np.float32, want.size), want)
    assert np.array_equal(p2.read(np.uint8, nxb), p1.read(np.uint8, nxb))
    for a in (wg, wu, xd, ws, g, u, o1, o2, o3, p1, p2):
        a.close()


# a clipped tile in both directions, a row count that is no multiple of four, one to three super-blocks, a bias
@pytest.mark.parametrize("tokens,out_dim,in_dim,with_bias", [(130, 25001, 256, True), (250, 24832, 512, False), (129, 24580, 768, True)])
def test_q6_k(gpu, oracle, tokens, out_dim, in_dim, with_bias, monkeypatch):
    rng = np.random.default_rng(out_dim)
    raw = synth.make_weights(rng, Q6_K, out_dim, in_dim)
    x = synth.make_activations(rng, tokens, in_dim)
    bias = rng.standard_normal(out_dim).astype(np.float32) if with_bias else None
    assert quant.gemm_plan(Q6_K, in_dim, out_dim, tokens, quant.gemm_workspace_bytes(Q6_K, in_dim, tokens))[0] == "q6_k_gemm_wide_f16"
    got = check(oracle, raw, x, in_dim, out_dim, tokens, bias, "Q6_K wide M=%d" % tokens, sample_tokens=[0, 31, 127, 128, tokens - 1], t=Q6_K)
    monkeypatch.setenv("COGNI_GEMM_WIDE", "0")
    assert np.array_equal(run_gemm(raw, x, in_dim, out_dim, tokens, bias, t=Q6_K).reshape(tokens, out_dim), got)


def test_q6_k_codes_and_scales_one_at_a_time(gpu, monkeypatch):
    """Every sub-block scale of both halves alone, against the four-wavefront kernel; residual in the epilogue."""
    monkeypatch.setenv("COGNI_GEMM_WIDE", "1")
    tokens, out_dim, in_dim = 96, 4096, 256
    rng = np.random.default_rng(61)
    x = synth.make_activations(rng, tokens, in_dim)
    for which in range(16):
        raw = synth.make_weights(rng, Q6_K, out_dim, in_dim).reshape(out_dim, 210)
        raw[:, 192:208] = 0
        raw[:, 192 + which] = np.uint8(256 - 7 * (which + 1) if which & 1 else 7 * (which + 1))
        raw = np.ascontiguousarray(raw.reshape(-1))
        assert quant.gemm_plan(Q6_K, in_dim, out_dim, tokens, quant.gemm_workspace_bytes(Q6_K, in_dim, tokens))[0] == "q6_k_gemm_wide_f16"
        wide = run_gemm(raw, x, in_dim, out_dim, tokens, t=Q6_K, split=False)
        monkeypatch.setenv("COGNI_GEMM_WIDE", "0")
        assert np.array_equal(run_gemm(raw, x, in_dim, out_dim, tokens, t=Q6_K, split=False), wide), which
        monkeypatch.setenv("COGNI_GEMM_WIDE", "1")
