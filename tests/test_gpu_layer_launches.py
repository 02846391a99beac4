"""Launches that do the work of several in a layer: each gives, bit for bit, what the separate launches give."""
import numpy as np
import pytest

from cogni_ml_amd import quant, synth
from gpu_common import DevArray, gpu  # noqa: F401
from helpers import Q4_K, Q5_K, Q6_K, Q8_0

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


@pytest.mark.parametrize("t", [Q4_K, Q5_K])
@pytest.mark.parametrize("in_dim,dims", [(4096, [4096, 1024, 1024, 12288, 12288]), (256, [1, 7, 3, 2]), (12288, [40, 9, 300, 5, 17, 2]),
                                         (2048, [9000, 1, 1, 1, 1, 1, 33])])
def test_lists_of_one_token(gpu, t, in_dim, dims):
    """Up to six matrices in a launch: each row as cogni_gemv_dev computes it."""
    rng = np.random.default_rng(in_dim + len(dims))
    xd = DevArray(synth.make_activations(rng, 1, in_dim))
    wd = [DevArray(synth.make_weights(rng, t, d, in_dim)) for d in dims]
    one, lst = ([DevArray(np.full(d, np.float32(5.0))) for d in dims] for _ in range(2))
    for w, o, d in zip(wd, one, dims):
        quant.gemv_dev(w.ptr, t, xd.ptr, o.ptr, in_dim, d)
    quant.gemv_many_dev([w.ptr for w in wd], t, xd.ptr, [o.ptr for o in lst], dims, in_dim)
    for a, b, d in zip(one, lst, dims):
        assert np.array_equal(a.read(np.float32, d), b.read(np.float32, d)), d
    for a in [xd] + wd + one + lst:
        a.close()


# both orders, both row counts per wavefront, rows of one and of several column sets, types without the kernel
@pytest.mark.parametrize("a,b", [((Q4_K, 4096, 4096), (Q6_K, 12288, 4096)), ((Q6_K, 3072, 1024), (Q5_K, 1024, 1024)), ((Q4_K, 8192, 3), (Q4_K, 256, 5000)),
                                 ((Q5_K, 2560, 2041), (Q4_K, 256, 2048)), ((Q6_K, 512, 40), (Q6_K, 256, 33)), ((Q4_K, 256, 1), (Q6_K, 256, 12300))])
def test_two_matrices_with_an_input_each(gpu, a, b):
    rng = np.random.default_rng(a[2] + b[2])
    mats = []
    for t, in_dim, out_dim in (a, b):
        mats.append((DevArray(synth.make_weights(rng, t, out_dim, in_dim)), t, DevArray(synth.make_activations(rng, 1, in_dim)),
                     DevArray(np.full(out_dim, np.float32(5.0))), DevArray(np.full(out_dim, np.float32(6.0))), in_dim, out_dim))
    for w, t, x, one, two, in_dim, out_dim in mats:
        quant.gemv_dev(w.ptr, t, x.ptr, one.ptr, in_dim, out_dim)
    quant.gemv_two_dev(*[v for w, t, x, one, two, in_dim, out_dim in mats for v in (w.ptr, t, x.ptr, two.ptr, in_dim, out_dim)])
    for w, t, x, one, two, in_dim, out_dim in mats:
        assert np.array_equal(one.read(np.float32, out_dim), two.read(np.float32, out_dim)), (t, in_dim, out_dim)
    w, t, x, one, two, in_dim, out_dim = mats[0]
    with pytest.raises(quant.QuantError, match="null device pointer"):
        quant.gemv_two_dev(w.ptr, t, 0, two.ptr, in_dim, out_dim, w.ptr, t, x.ptr, two.ptr, in_dim, out_dim)
    for m in mats:
        for i in (0, 2, 3, 4):
            m[i].close()


# lists whose tile counts take one, two and three tiles per wavefront, a ragged last matrix, streamed operands, sixteen tokens
@pytest.mark.parametrize("t", [Q4_K, Q5_K])
@pytest.mark.parametrize("tokens,in_dim,dims", [(8, 4096, [4096, 1024, 1024, 12288, 12288]), (2, 2048, [16, 32, 48, 5]), (5, 1024, [4096, 16, 6000, 160, 11]),
                                                (3, 6144, [16, 160, 32, 48, 64, 9]), (16, 2048, [1024, 256, 256, 9008, 7]), (9, 12288, [16, 16, 16, 40])])
def test_lists_of_several_tokens(gpu, t, tokens, in_dim, dims):
    """Four to six matrices against one image: each output as the image and that matrix alone give it."""
    rng = np.random.default_rng(in_dim + tokens)
    pack, packed = (quant.gemv_pack16_dev, quant.gemv_packed16_dev) if tokens > 8 else (quant.gemv_pack_dev, quant.gemv_packed_dev)
    xd, image = DevArray(synth.make_activations(rng, tokens, in_dim)), DevArray(nbytes=quant.gemv_image_bytes(t, in_dim, 8))
    wd = [DevArray(synth.make_weights(rng, t, d, in_dim)) for d in dims]
    one, lst = ([DevArray(np.full(tokens * d, np.float32(5.0))) for d in dims] for _ in range(2))
    pack(xd.ptr, t, in_dim, tokens, image.ptr)
    for w, o, d in zip(wd, one, dims):
        packed([w.ptr], t, image.ptr, [o.ptr], [d], in_dim, tokens)
    packed([w.ptr for w in wd], t, image.ptr, [o.ptr for o in lst], dims, in_dim, tokens)
    for a, b, d in zip(one, lst, dims):
        assert np.array_equal(a.read(np.float32, tokens * d), b.read(np.float32, tokens * d)), d
    for a in [xd, image] + wd + one + lst:
        a.close()


@pytest.mark.parametrize("kind", ["gemv", "gemv16", "gemm"])
@pytest.mark.parametrize("a,b", [((Q4_K, 4096), (Q6_K, 12288)), ((Q6_K, 256), (Q5_K, 2816)), ((Q4_K, 512), (Q4_K, 256))])
def test_two_activation_blocks_in_one_launch(gpu, kind, a, b):
    tokens = {"gemv": 5, "gemv16": 13, "gemm": 130}[kind]
    rng = np.random.default_rng(a[1] + b[1])
    args, blocks = [], []
    for t, in_dim in (a, b):
        x = DevArray(synth.make_activations(rng, tokens, in_dim))
        nb = quant.gemm_workspace_bytes(t, in_dim, tokens) if kind == "gemm" else quant.gemv_image_bytes(t, in_dim, 8)
        p, q = (DevArray(np.full(nb, 0xFF, np.uint8)) for _ in range(2))
        if kind == "gemm":
            quant.gemm_pack_dev(x.ptr, t, in_dim, tokens, p.ptr, nb)
            args += [x.ptr, t, in_dim, q.ptr, nb]
        else:
            (quant.gemv_pack_dev if kind == "gemv" else quant.gemv_pack16_dev)(x.ptr, t, in_dim, tokens, p.ptr)
            args += [x.ptr, t, in_dim, q.ptr]
        blocks.append((x, p, q, nb))
    {"gemv": quant.gemv_pack_two_dev, "gemv16": quant.gemv_pack16_two_dev, "gemm": quant.gemm_pack_two_dev}[kind](*args, tokens)
    for x, p, q, nb in blocks:
        assert np.array_equal(p.read(np.uint8, nb), q.read(np.uint8, nb))
        for d in (x, p, q):
            d.close()


def test_rounds_of_a_stack():
    """What reads an output comes in a later round; what cannot be put into rounds stays in its order."""
    from cogni_ml_amd.projection_stack import QWEN_LAYER_4096, QwenProjectionStackRunner
    rounds = QwenProjectionStackRunner._rounds_of([e + (None,) for e in QWEN_LAYER_4096])
    assert [[[e[0] for e in g] for g in r] for r in rounds] == [[["q", "k", "v", "gate", "up"]], [["o"], ["down"]]]
    for odd in ([("a", "b", Q4_K, 256, 256, None), ("b", "x", Q4_K, 256, 256, None)], [("a", "x", Q4_K, 256, 256, None), ("a", "x", Q4_K, 256, 256, None)]):
        assert QwenProjectionStackRunner._rounds_of(odd) == [[[e]] for e in odd]


# both orders, one and six super-blocks per k-slice, rows past the grid's 256 tiles, a ragged end, pairs without a kernel (two tiles a wavefront, types)
@pytest.mark.parametrize("tokens", [2, 7, 8, 9, 16])
@pytest.mark.parametrize("a,b", [((Q4_K, 4096, 4096), (Q6_K, 12288, 4096)), ((Q6_K, 2816, 1000), (Q5_K, 1024, 1024)), ((Q4_K, 256, 1), (Q4_K, 8192, 5000)),
                                 ((Q5_K, 5376, 33), (Q4_K, 2560, 16)), ((Q4_K, 1024, 12288), (Q6_K, 256, 70)), ((Q6_K, 512, 40), (Q6_K, 256, 33))])
def test_two_matrices_with_an_image_each(gpu, a, b, tokens):
    """The launch of two matrices: each output as its image and that matrix alone give it, bit for bit."""
    x16 = tokens > 8
    pack, packed, two = (quant.gemv_pack16_dev, quant.gemv_packed16_dev, quant.gemv_packed16_two_dev) if x16 else \
        (quant.gemv_pack_dev, quant.gemv_packed_dev, quant.gemv_packed_two_dev)
    rng = np.random.default_rng(a[1] + b[1] + tokens)
    args, mats = [], []
    for t, in_dim, out_dim in (a, b):
        x, image = DevArray(synth.make_activations(rng, tokens, in_dim)), DevArray(nbytes=quant.gemv_image_bytes(t, in_dim, 8))
        w = DevArray(synth.make_weights(rng, t, out_dim, in_dim))
        one, both = (DevArray(np.full(tokens * out_dim + 64, np.float32(v))) for v in (5.0, 6.0))
        pack(x.ptr, t, in_dim, tokens, image.ptr)
        packed([w.ptr], t, image.ptr, [one.ptr], [out_dim], in_dim, tokens)
        args += [w.ptr, t, image.ptr, both.ptr, in_dim, out_dim]
        mats.append((x, image, w, one, both, out_dim))
    print("case", a, b, tokens, flush=True)
    two(*args, tokens)
    for x, image, w, one, both, out_dim in mats:
        got = both.read(np.float32, tokens * out_dim + 64)
        assert np.array_equal(got[:tokens * out_dim], one.read(np.float32, tokens * out_dim)), out_dim
        assert (got[tokens * out_dim:] == 6.0).all()
    with pytest.raises(quant.QuantError, match="null pointer"):
        two(*args[:3], 0, *args[4:], tokens)
    for m in mats:
        for d in m[:5]:
            d.close()


@pytest.mark.parametrize("in_dim", [256, 768, 2048, 3328, 4096, 12288])
@pytest.mark.parametrize("first", [0, 1, 2, 3, 4, 10, 14, 15])
def test_q6_k_blocks_at_every_shift(gpu, oracle, first, in_dim):
    """The one-pass kernels copy a Q6_K block as the aligned 16-byte pieces that hold it: rows of odd and even numbers of blocks (blocks
    inside and at the start of a dword), and a matrix that starts `first` bytes behind 16 aligned ones."""
    out_dim, tokens = 37, 5
    rng = np.random.default_rng(in_dim + first)
    raw, x = synth.make_weights(rng, Q6_K, out_dim, in_dim), synth.make_activations(rng, tokens, in_dim)
    w = DevArray(np.concatenate([np.full(first, 0x5A, np.uint8), np.frombuffer(raw, np.uint8), np.full(16, 0xA5, np.uint8)]))
    xd, image = DevArray(x), DevArray(nbytes=quant.gemv_image_bytes(Q6_K, in_dim, 8))
    od = DevArray(np.full(tokens * out_dim, np.nan, dtype=np.float32))
    quant.gemv_pack_dev(xd.ptr, Q6_K, in_dim, tokens, image.ptr)
    quant.gemv_packed_dev([w.ptr + first], Q6_K, image.ptr, [od.ptr], [out_dim], in_dim, tokens)
    got = od.read(np.float32, tokens * out_dim)
    want = oracle.matmul_add(x, tokens, in_dim, raw, Q6_K, out_dim, np.zeros(out_dim, dtype=np.float32))
    # the bound of smoke(): 22-bit activations and fp32 sums against 64 bits
    tol = 1e-4 * np.linalg.norm(x.reshape(tokens, -1), axis=1).max() * np.abs(oracle.dequantize(raw, Q6_K, out_dim * in_dim)).max()
    assert np.abs(got - want).max() <= tol and np.linalg.norm(got - want) <= 1e-5 * np.linalg.norm(want)
    for d in (w, xd, image, od):
        d.close()


# row counts on both sides of the rule's lines: one tile in several rounds, two and three tiles, a last group that is not full
@pytest.mark.parametrize("rows", [4097, 8200, 13386, 24577])
@pytest.mark.parametrize("t,in_dim", [(Q4_K, 1024), (Q5_K, 1536), (Q6_K, 768), (Q6_K, 1024), (Q6_K, 2048), (Q6_K, 3328), (Q8_0, 1024)])
def test_rows_do_not_depend_on_the_tiles_per_wavefront(gpu, t, in_dim, rows):
    """Every row as from launches of up to 256 tiles of 16 rows, which take one tile per wavefront; up to eight tokens and sixteen."""
    rng = np.random.default_rng(rows + in_dim)
    raw = synth.make_weights(rng, t, rows, in_dim)
    row_bytes, part = len(raw) // rows, 4096
    w, x = DevArray(raw), DevArray(synth.make_activations(rng, 13, in_dim))
    image = DevArray(nbytes=quant.gemv_image_bytes(t, in_dim, 8))
    for tokens, pack, gemv in ((7, quant.gemv_pack_dev, quant.gemv_packed_dev), (13, quant.gemv_pack16_dev, quant.gemv_packed16_dev)):
        out = DevArray(np.full(tokens * rows, np.nan, np.float32))
        pack(x.ptr, t, in_dim, tokens, image.ptr)
        gemv([w.ptr], t, image.ptr, [out.ptr], [rows], in_dim, tokens)
        got = out.read(np.float32, tokens * rows).reshape(tokens, rows)
        for r0 in range(0, rows, part):
            n = min(part, rows - r0)
            piece = DevArray(np.full(tokens * n, np.nan, np.float32))
            gemv([w.ptr + r0 * row_bytes], t, image.ptr, [piece.ptr], [n], in_dim, tokens)
            assert np.array_equal(piece.read(np.float32, tokens * n).reshape(tokens, n), got[:, r0:r0 + n]), r0
            piece.close()
        out.close()
    for d in (w, x, image):
        d.close()
