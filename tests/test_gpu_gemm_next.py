"""Prefill lists that leave outputs as the packed inputs of following GEMMs: outputs and packed bytes, and the runner that goes by them."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from cogni_ml_amd.projection_stack import QwenProjectionStackRunner, Weights
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K

pytestmark = pytest.mark.gpu


# both kernels, tokens that end inside a tile of 32, of 64, of 128, of 256, or with it; a list with one packed output, several, of both layouts, beside
# matrices of odd row counts; rows that end a workgroup's tile inside a matrix (256 and 512 rows of tiles of 32, 64 and 256)
@pytest.mark.parametrize("kernel,w_type,tokens,in_dim,dims,nexts", [
    ("stream", Q4_K, 17, 256, [256, 7], [Q6_K, None]), ("stream", Q4_K, 32, 512, [512, 256, 33], [Q4_K, Q6_K, None]),
    ("stream", Q4_K, 33, 1024, [100, 256, 512], [None, Q4_K, Q6_K]), ("stream", Q4_K, 64, 256, [8192, 8192], [Q6_K, Q4_K]),
    ("stream", Q4_K, 129, 512, [256] * 6, [Q4_K] * 6), ("stream", Q5_K, 20, 256, [256, 768], [Q4_K, Q6_K]),
    ("stream", Q5_K, 75, 512, [512, 64], [Q6_K, None]), ("tall", Q4_K, 129, 256, [256, 300], [Q6_K, None]),
    ("tall", Q4_K, 256, 512, [65, 512, 256], [None, Q4_K, Q6_K]), ("tall", Q4_K, 400, 768, [768], [Q4_K]),
    ("tall", Q4_K, 513, 256, [256, 256], [Q6_K, Q4_K]), ("tall", Q4_K, 1, 256, [256], [Q6_K])])
def test_lists_with_packed_outputs(gpu, kernel, w_type, tokens, in_dim, dims, nexts):
    """The outputs are those of the list without packed inputs, bit for bit, and the packed bytes those of a pack of the outputs (of the tokens there
    are and, tall, the absent ones)."""
    plain, pack = (quant.gemm_tall_dev, quant.gemm_tall_pack_dev) if kernel == "tall" else (quant.gemm_stream_dev, quant.gemm_stream_pack_dev)
    rng = np.random.default_rng(tokens * 7 + in_dim)
    x, ws = DevArray(synth.make_activations(rng, tokens, in_dim)), DevArray(nbytes=quant.gemm_workspace_bytes(w_type, in_dim, tokens))
    wsb = quant.gemm_workspace_bytes(w_type, in_dim, tokens)
    wd = [DevArray(synth.make_weights(rng, w_type, d, in_dim)) for d in dims]
    outs = [[DevArray(np.full(tokens * d + 4, np.float32(-3.0))) for d in dims] for _ in range(2)]
    size = [quant.gemm_workspace_bytes(t, d, tokens) if t else 0 for t, d in zip(nexts, dims)]
    got, want = ([DevArray(np.full(n + 64, 0xFF, np.uint8)) if n else None for n in size] for _ in range(2))
    quant.gemm_pack_dev(x.ptr, w_type, in_dim, tokens, ws.ptr, wsb)
    w = [a.ptr for a in wd]
    plain(w, w_type, ws.ptr, wsb, [o.ptr for o in outs[0]], dims, in_dim, tokens)
    pack(w, w_type, ws.ptr, wsb, [o.ptr for o in outs[1]], dims, [(t, g.ptr, n) if t else None for t, g, n in zip(nexts, got, size)], in_dim, tokens)
    for a, b, d in zip(*outs, dims):
        assert np.array_equal(a.read(np.uint32, tokens * d + 4), b.read(np.uint32, tokens * d + 4)), d
    for t, o, g, p, d, n in zip(nexts, outs[1], got, want, dims, size):
        if not t:
            continue
        quant.gemm_pack_dev(o.ptr, t, d, tokens, p.ptr, n)
        a, b = (v.read(np.uint8, n + 64) for v in (g, p))
        assert np.all(a[n:] == 0xFF)
        a, b = (v[:n].reshape(-1, d // 256, 32, 128, 16) for v in (a, b))   # [128-token tile][super-block][cell][token]
        a, b = (np.moveaxis(v, 3, 1).reshape(v.shape[0] * 128, -1) for v in (a, b))
        written = len(a) if kernel == "tall" else -(-tokens // 32) * 32
        assert np.array_equal(a[:written], b[:written]), d
    for a in [x, ws] + wd + sum(outs, []) + [v for v in got + want if v]:
        a.close()


@pytest.mark.parametrize("tokens,w_type,down", [(40, Q4_K, Q6_K), (40, Q5_K, Q4_K), (400, Q4_K, Q6_K)])
def test_runner_of_packed_outputs(gpu, tokens, w_type, down, monkeypatch):
    """The runner with and without them: the same bits, and without is what it does when no list writes one."""
    rng = np.random.default_rng(tokens)
    weights = Weights.synthetic(rng, [("q", "x", w_type, 2048, 2048), ("k", "x", w_type, 512, 2048), ("gate", "x", w_type, 14336, 2048),
                                      ("up", "x", w_type, 14336, 2048), ("o", "q", w_type, 2048, 2048), ("down", "up", down, 2048, 14336)])
    xs = synth.make_activations(rng, tokens, 2048).reshape(-1)
    seen = []
    for name in ("gemm_stream_pack_dev", "gemm_tall_pack_dev"):
        f = getattr(quant, name)
        monkeypatch.setattr(quant, name, lambda *a, f=f, name=name: (seen.append(name), f(*a))[1])
    results = []
    for without in (False, True):
        if without:
            monkeypatch.setattr(QwenProjectionStackRunner, "_next_input", lambda self, e: None)
        r = QwenProjectionStackRunner.from_weights(weights, tokens, xs)
        r.upload_weights()
        for _ in range(3):   # as it is written, noted, from the notes
            r.reset_sequence()
            r.run_sequence()
        r.read_outputs()
        results.append({k: v.view(np.uint32).copy() for k, v in r.outputs.items()})
        r.close()
    assert len(seen) == 2, seen
    for k in results[0]:
        assert np.array_equal(results[0][k], results[1][k]), k


def test_a_first_pass_asks_no_more_than_it_needs(gpu, monkeypatch):
    """What a prefill of any length has to know of the projections is found when the runner is made, and a short prefill asks for none of the tiles of many tokens."""
    rng = np.random.default_rng(3)
    weights = Weights.synthetic(rng, [("q", "x", Q4_K, 2048, 2048), ("k", "x", Q4_K, 512, 2048), ("gate", "x", Q4_K, 11008, 2048), ("up", "x", Q4_K, 11008, 2048),
                                      ("o", "q", Q4_K, 2048, 2048), ("down", "up", Q6_K, 2048, 11008)])
    r = QwenProjectionStackRunner.from_weights(weights, 512, synth.make_activations(rng, 512, 2048).reshape(-1))
    assert r._two_scratch is not None
    asked = []
    for owner, name in ((quant, "gemm_tall_takes"), (quant, "gemm_wide_two_takes"), (quant, "gemv_image_bytes"), (QwenProjectionStackRunner, "_next_input")):
        f = getattr(owner, name)
        monkeypatch.setattr(owner, name, lambda *a, f=f, name=name: (asked.append(name), f(*a))[1])
    r.upload_weights()
    r.reset_sequence()
    for count, want in ((48, []), (512, ["gemm_tall_takes", "gemm_wide_two_takes"])):
        r.active_tokens = count
        r.run_sequence()
        assert asked == want, count
    r.read_outputs()
    r.close()


def test_refusals(gpu):
    bad = [([256, 256], [(Q6_K, 64, 1 << 30), None], Q6_K, "Unsupported quant type"), ([300], [(Q6_K, 64, 1 << 30)], Q4_K, "multiple of 256"),
           ([256], [(Q6_K, 64, 16)], Q4_K, "next_workspace too small"), ([256], [(8, 64, 1 << 30)], Q4_K, "Unsupported quant type")]
    for f in (quant.gemm_stream_pack_dev, quant.gemm_tall_pack_dev):
        for dims, nexts, t, match in bad:
            with pytest.raises(quant.QuantError, match=match):
                f([64] * len(dims), t, 64, 1 << 30, [64] * len(dims), dims, nexts, 256, 200)
        with pytest.raises(ValueError, match="one entry per matrix"):
            f([64], Q4_K, 64, 1 << 30, [64], [256], [], 256, 200)
