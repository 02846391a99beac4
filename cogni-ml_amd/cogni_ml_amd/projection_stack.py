"""Resident decoder-layer projection stack on one HIP stream.

The HIP counterpart of the reference's resident projection runners
(src/ml/cuda/qwen_full_attn_projection_runner.cr: q/k/v bundle; bin/cuda_ffn_sequence_probe.cr:
gate/up/down): weights and activations stay on the device, every projection of every token group is
launched back to back into the current stream, and the lifecycle goes through ResidentSequenceRunner
(upload_weights -> reset_sequence -> run_sequence x reps -> synchronize -> read_outputs).

Where the reference runs either one launch per token or weight-stationary groups of 4 tokens
(`tbatch4`, qwen_full_attn_projection_runner.cr:274-301), this runner hands groups of up to 8 tokens
to one weight-stationary launch. A sequence of more tokens than the GEMM threshold (quant.get_gemm_threshold(), 8 as
in the reference's router) goes through the prefill GEMMs instead, all tokens at once: every distinct input is packed
once (q | k | v and gate | up share x) and each projection is one GEMM against it - the reference's
`qmatmul_nobias(qw, x, batch)` calls of a prefill layer (src/ml/gguf/qwen35_cpu.cr:1478-1490).
"""
import collections

import numpy as np

from . import hip, quant
from .types import TensorType

# (name, input, weight type, out_dim, in_dim) at the shapes of the benchmark's mixed-quant layer:
# hidden 4096, 32 query / 8 KV heads of 128, FFN 12288; q/k/v/o/gate/up Q4_K, down Q6_K
QWEN_LAYER_4096 = [
    ("q", "x", TensorType.Q4_K, 4096, 4096),
    ("k", "x", TensorType.Q4_K, 1024, 4096),
    ("v", "x", TensorType.Q4_K, 1024, 4096),
    ("o", "q", TensorType.Q4_K, 4096, 4096),
    ("gate", "x", TensorType.Q4_K, 12288, 4096),
    ("up", "x", TensorType.Q4_K, 12288, 4096),
    ("down", "gate", TensorType.Q6_K, 4096, 12288),
]


class Weights:
    """Raw GGUF bytes per projection: {name: (raw, type, out_dim, in_dim, input name)}."""

    def __init__(self, hidden, entries):
        self.hidden = hidden
        self.entries = entries        # ordered list of (name, input, type, out_dim, in_dim, raw)

    @classmethod
    def synthetic(cls, rng, layout=QWEN_LAYER_4096):
        from . import synth
        hidden = layout[0][4]
        return cls(hidden, [(n, src, t, o, i, synth.make_weights(rng, t, o, i)) for n, src, t, o, i in layout])

    @property
    def raw_bytes(self):
        return sum(e[5].size for e in self.entries)


# a group of projections as a prefill launches it (the first field is the name of its first projection, as in Weights.entries)
PrefillGroup = collections.namedtuple("PrefillGroup", "name key type in_dim x ws nbytes image16 lists w out dims nexts entry")


class QwenProjectionStackRunner:
    def __init__(self, weights, tokens, xs):
        if not tokens > 0:
            raise ValueError("tokens must be positive")
        if len(xs) != tokens * weights.hidden:
            raise ValueError("xs size mismatch")
        self.weights, self.tokens, self.hidden = weights, tokens, weights.hidden
        self._xs = np.ascontiguousarray(xs, dtype=np.float32)
        self._buffers = []
        self._rounds = self._rounds_of(weights.entries)
        self._w = {}
        self._images = {}   # (input name, weight type) -> packed activation image shared by every list that reads that input
        self._act = {"x": self._alloc(4 * tokens * self.hidden)}
        for name, src, t, out_dim, in_dim, raw in weights.entries:
            self._w[name] = self._alloc(raw.size)
            self._act[name] = self._alloc(4 * tokens * out_dim)
            # (allocated here, not at first use: the sequence may be issued under stream capture)
            nbytes = quant.gemv_image_bytes(t, in_dim, quant.MAX_GEMV_TOKENS)
            if nbytes and (src, int(t)) not in self._images:
                self._images[(src, int(t))] = self._alloc(nbytes)
        # prefill: one workspace per (input, packed layout) - Q4_K and Q5_K read one layout, Q6_K its own - large enough
        # for the k-split planes of the projection that needs the most
        self._prefill_ws = {}
        self._images16 = {}   # input name -> the image of the sixteen-token one-pass kernels (Q4_K / Q5_K projections, 9..16 tokens)
        if tokens > quant.get_gemm_threshold() and all(self._gemm_capable(e) for e in weights.entries):
            need = {}
            for name, src, t, out_dim, in_dim, raw in weights.entries:
                key = (src, self._family(t))
                need[key] = max(need.get(key, 0), quant.gemm_workspace_bytes(t, in_dim, tokens, out_dim))
                if self._one_pass16(t, in_dim) and key not in self._images16:
                    self._images16[key] = self._alloc(quant.gemv_image_bytes(t, in_dim, quant.MAX_GEMV_TOKENS))
            self._prefill_ws = {k: (self._alloc(n), n) for k, n in need.items()}
        # planes of two single matrices that share a launch, allocated where some token count may take it
        self._two_scratch = self._alloc(quant.gemm_wide_two_scratch_bytes()) if self._prefill_ws and any(
            self._wide_two(g[0], h[0], n) for groups in self._rounds for i, g in enumerate(groups) for h in groups[i + 1:] if len(g) == len(h) == 1
            for n in [tokens, *range(193, tokens, 64)]) else None
        self._prefill_groups = [[self._prefill_group(g) for g in groups] for groups in self._rounds] if self._prefill_ws else []
        self._issued = {}   # prefill: the library calls of a token count
        self.outputs = {}
        self._runner = hip.ResidentSequenceRunner(
            tokens, self._upload_weights, self._reset_sequence, self._run_token, self._read_outputs,
            self._run_sequence)

    @classmethod
    def from_weights(cls, weights, tokens, xs):
        return cls(weights, tokens, xs)

    def _alloc(self, nbytes):
        b = hip.DeviceBuffer(nbytes)
        self._buffers.append(b)
        return b

    # ---- closures handed to ResidentSequenceRunner -------------------------------------------------
    def _upload_weights(self):
        for name, src, t, out_dim, in_dim, raw in self.weights.entries:
            hip.copy_htod(self._w[name].ptr, raw, raw.size, "%s weights" % name)

    def _reset_sequence(self):
        hip.copy_htod(self._act["x"].ptr, self._xs, self._xs.nbytes, "sequence input")

    @staticmethod
    def _rounds_of(entries):
        """The projections in rounds: one that reads another's output is in a later round than that, so the projections of a round
        are independent of each other. A round is a list of groups of up to six that share input, type and row length (q | k | v |
        gate | up), each group one launch."""
        depth, rounds = {"x": 0}, []
        for e in entries:
            name, src, t, out_dim, in_dim, raw = e
            if src not in depth or name in depth:   # reads what a later one writes, or writes a buffer again: strictly in order
                return [[[e]] for e in entries]
            d = depth[name] = depth[src] + 1
            while len(rounds) < d:
                rounds.append([])
            for grp in rounds[d - 1]:
                if len(grp) < 6 and (grp[0][1], int(grp[0][2]), grp[0][4]) == (src, int(t), in_dim):
                    grp.append(e)
                    break
            else:
                rounds[d - 1].append([e])
        return rounds

    @staticmethod
    def _pack_each(jobs, one, two):
        """The activation blocks of `jobs`, two to a launch."""
        for i in range(0, len(jobs) - 1, 2):
            two(*jobs[i], *jobs[i + 1])
        if len(jobs) % 2:
            one(*jobs[-1])

    @staticmethod
    def _pairs(entries, two):
        """Entries that are launched alone go two to a launch; the names that have been."""
        n = len(entries) // 2 * 2
        for i in range(0, n, 2):
            two(entries[i], entries[i + 1])
        return {e[0] for e in entries[:n]}

    def _launch(self, tok0, count):
        stream = hip.current_stream_handle()

        def act(name, dim):
            return self._act[name].ptr + 4 * tok0 * dim

        for groups in self._rounds:
            # several tokens of a shape the one-pass kernel takes: every input is packed once, and what reads it goes against that
            # image; the others through the library, which picks their kernels
            imaged, singles, jobs = [], [], {}
            for grp in groups:
                name, src, t, out_dim, in_dim, raw = grp[0]
                start = quant.gemv_one_pass_multi_from(t, in_dim) if len(grp) >= 2 else quant.gemv_one_pass_from(t, in_dim, out_dim)
                if 1 < count and 0 < start <= count:
                    jobs.setdefault((src, int(t)), (act(src, in_dim), t, in_dim, self._images[(src, int(t))].ptr))
                    imaged.append(grp)
                elif len(grp) >= 2:
                    most = 6 if count == 1 else 3   # matrices in a launch of the kernels for one and for several tokens
                    for part in (grp[i:i + most] for i in range(0, len(grp), most)):
                        quant.gemv_many_dev([self._w[e[0]].ptr for e in part], t, act(src, in_dim), [act(e[0], e[3]) for e in part],
                                            [e[3] for e in part], in_dim, count, stream)
                else:
                    singles.append((self._w[name].ptr, t, act(src, in_dim), act(name, out_dim), in_dim, out_dim))
            self._pack_each(list(jobs.values()), lambda x, t, k, image: quant.gemv_pack_dev(x, t, k, count, image, stream),
                            lambda *ab: quant.gemv_pack_two_dev(*ab, count, stream))
            def one_image(e):
                name, src, t, out_dim, in_dim, raw = e
                return self._w[name].ptr, t, self._images[(src, int(t))].ptr, act(name, out_dim), in_dim, out_dim

            done = self._pairs([g[0] for g in imaged if len(g) == 1],
                               lambda a, b: quant.gemv_packed_two_dev(*one_image(a), *one_image(b), count, stream))
            for grp in imaged:
                if grp[0][0] in done:
                    continue
                name, src, t, out_dim, in_dim, raw = grp[0]
                quant.gemv_packed_dev([self._w[e[0]].ptr for e in grp], t, self._images[(src, int(t))].ptr, [act(e[0], e[3]) for e in grp],
                                      [e[3] for e in grp], in_dim, count, 0, stream)
            for i in range(0, len(singles) - 1, 2):
                quant.gemv_two_dev(*singles[i], *singles[i + 1], count, stream)
            if len(singles) % 2:
                w, t, x, out, in_dim, out_dim = singles[-1]
                quant.gemv_dev(w, t, x, out, in_dim, out_dim, count, 0, stream)

    @staticmethod
    def _family(t):
        return "q6" if int(t) == int(TensorType.Q6_K) else "q45"

    @staticmethod
    def _wide_two(a, b, count):
        return quant.gemm_wide_two_takes(a[2], a[4], a[3], b[2], b[4], b[3], count)

    @staticmethod
    def _gemm_capable(entry):
        return int(entry[2]) in (int(TensorType.Q4_K), int(TensorType.Q5_K), int(TensorType.Q6_K)) and entry[4] % 256 == 0

    @staticmethod
    def _one_pass16(t, in_dim):
        return int(t) in (int(TensorType.Q4_K), int(TensorType.Q5_K), int(TensorType.Q6_K)) and \
            quant.gemv_image_bytes(t, in_dim, quant.MAX_GEMV_TOKENS) > 0

    def _next_input(self, entry):
        """What a list can write beside this output: ((output name, layout), (type, workspace, bytes)) of a projection that reads it."""
        for name, src, t, out_dim, in_dim, raw in self.weights.entries:
            if src == entry[0] and in_dim == entry[3]:
                ws, nbytes = self._prefill_ws[(src, self._family(t))]
                return (src, self._family(t)), (t, ws.ptr, nbytes)
        return None

    def _prefill_group(self, grp):
        """What a prefill of any token count has to know of a group of a round."""
        name, src, t, out_dim, in_dim, raw = grp[0]
        key = (src, self._family(t))
        ws, nbytes = self._prefill_ws[key]
        lists = int(t) in (int(TensorType.Q4_K), int(TensorType.Q5_K))
        nexts = [self._next_input(e) for e in grp] if len(grp) >= 2 and lists else []
        return PrefillGroup(name=name, key=key, type=t, in_dim=in_dim, x=self._act[src].ptr, ws=ws.ptr, nbytes=nbytes,
                            image16=self._images16[key].ptr if self._one_pass16(t, in_dim) else None, lists=lists,
                            w=[self._w[e[0]].ptr for e in grp], out=[self._act[e[0]].ptr for e in grp], dims=[e[3] for e in grp],
                            nexts=nexts if any(nexts) else [], entry=grp[0])

    def _launch_prefill(self, count):
        """All `count` tokens through the GEMMs: one pack per (input, layout), one GEMM per list of projections that share
        their input, type and row length (or per projection). A list that can leaves its outputs as the packed inputs of the
        rounds behind it too."""
        stream = hip.current_stream_handle()
        packed = set()   # the (input, layout) that a list has written

        # single matrices of up to sixteen tokens, or of short prefills, or two that share the chip: two to a launch (o and down)
        def one_image(g):
            return g.w[0], g.type, g.image16, g.out[0], g.in_dim, g.dims[0]

        def one_packed(g):
            return g.w[0], g.type, g.ws, g.nbytes, g.out[0], g.in_dim, g.dims[0]

        for groups in self._prefill_groups:
            # the inputs of the round, packed once each, two to a launch
            jobs16, jobs = {}, {}
            for g in groups:
                if count <= 16 and g.image16:
                    jobs16.setdefault(g.key, (g.x, g.type, g.in_dim, g.image16))
                elif g.key not in packed:
                    jobs.setdefault(g.key, (g.x, g.type, g.in_dim, g.ws, g.nbytes))
            self._pack_each(list(jobs16.values()), lambda x, t, k, image: quant.gemv_pack16_dev(x, t, k, count, image, stream),
                            lambda *ab: quant.gemv_pack16_two_dev(*ab, count, stream))
            self._pack_each(list(jobs.values()), lambda x, t, k, ws, nbytes: quant.gemm_pack_dev(x, t, k, count, ws, nbytes, stream),
                            lambda *ab: quant.gemm_pack_two_dev(*ab, count, stream))
            alone = [g for g in groups if len(g.w) == 1]
            done = set()
            if len(alone) >= 2:
                done = self._pairs([g for g in alone if g.key in jobs16],
                                   lambda a, b: quant.gemv_packed16_two_dev(*one_image(a), *one_image(b), count, stream))
                if self._two_scratch is not None and count > 128:   # (tiles of 128 tokens)
                    for i, a in enumerate(alone):
                        b = next((g for g in alone[i + 1:] if g.name not in done and self._wide_two(a.entry, g.entry, count)), None)
                        if b is not None and a.name not in done:
                            quant.gemm_wide_two_dev(*one_packed(a), *one_packed(b), self._two_scratch.ptr, quant.gemm_wide_two_scratch_bytes(), count, stream)
                            done |= {a.name, b.name}
                done |= self._pairs([g for g in alone if g.key not in jobs16 and g.name not in done and
                                     quant.gemm_stream_takes(g.type, g.in_dim, g.dims[0], count)],
                                    lambda a, b: quant.gemm_stream_two_dev(*one_packed(a), *one_packed(b), count, stream))
            for g in groups:
                if g.name in done:
                    continue
                t, in_dim, w, out, dims, nexts = g.type, g.in_dim, g.w, g.out, g.dims, g.nexts
                if g.key in jobs16:
                    # up to sixteen tokens: the one-pass decode kernels with sixteen single-term tokens
                    quant.gemv_packed16_dev(w, t, g.image16, out, dims, in_dim, count, 0, stream)
                    continue
                while dims:   # (the prefill counterpart of the qmatvec_many seam)
                    takes = quant.gemm_stream_takes(t, in_dim, sum(dims), count)
                    tall = not takes and quant.gemm_tall_takes(t, in_dim, dims, count)
                    if nexts and (takes or tall):
                        (quant.gemm_stream_pack_dev if takes else quant.gemm_tall_pack_dev)(
                            w, t, g.ws, g.nbytes, out, dims, [n and n[1] for n in nexts], in_dim, count, stream)
                        packed.update(n[0] for n in nexts if n)
                        break
                    if takes:
                        quant.gemm_stream_dev(w, t, g.ws, g.nbytes, out, dims, in_dim, count, 0, stream)
                        break
                    if tall:
                        quant.gemm_tall_dev(w, t, g.ws, g.nbytes, out, dims, in_dim, count, stream)
                        break
                    if len(dims) >= 2 and g.lists:
                        quant.gemm_packed_many_dev(w, t, g.ws, g.nbytes, out, dims, in_dim, count, stream)
                        break
                    quant.gemm_packed_dev(w[0], t, g.ws, g.nbytes, out[0], in_dim, dims[0], count, 0, stream)
                    w, out, dims, nexts = w[1:], out[1:], dims[1:], nexts[1:]

    def _run_token(self, tok):
        self._launch(tok, 1)

    def _run_sequence(self, active_tokens):
        if self._prefill_ws and active_tokens > quant.get_gemm_threshold():
            hip.issue(self._issued, active_tokens, lambda: self._launch_prefill(active_tokens), quant._check)
            return
        for tok0 in range(0, active_tokens, quant.MAX_GEMV_TOKENS):
            self._launch(tok0, min(quant.MAX_GEMV_TOKENS, active_tokens - tok0))

    def _read_outputs(self):
        hip.synchronize("hipDeviceSynchronize(read_outputs)")
        for name, src, t, out_dim, in_dim, raw in self.weights.entries:
            out = np.empty(self.tokens * out_dim, dtype=np.float32)
            hip.copy_dtoh(out, self._act[name].ptr, out.nbytes, "%s output" % name)
            self.outputs[name] = out

    # ---- public lifecycle, as the reference runner's (qwen_full_attn_projection_runner.cr:111-165) ----
    def upload_weights(self):
        self._runner.upload_weights()

    def replace_sequence_input(self, xs):
        if len(xs) != self.tokens * self.hidden:
            raise ValueError("xs size mismatch")
        self._xs = np.ascontiguousarray(xs, dtype=np.float32)

    def reset_sequence(self):
        self._runner.reset_sequence()

    def run_sequence(self):
        self._runner.run_sequence()

    def run_repeated(self, reps):
        return self._runner.run_repeated(reps)

    @property
    def active_tokens(self):
        return self._runner.active_tokens

    @active_tokens.setter
    def active_tokens(self, count):
        self._runner.active_tokens = count

    def reset_active_tokens(self):
        self._runner.reset_active_tokens()

    def read_outputs(self):
        self._runner.read_outputs()

    def device_ptr(self, name):
        return self._act[name].ptr

    def bytes_per_sequence(self, active_tokens=None):
        """Algorithmic bytes of one run_sequence: every weight once per group of up to 8 tokens, x in, out out."""
        m = self.tokens if active_tokens is None else active_tokens
        groups = 1 if (self._prefill_ws and m > quant.get_gemm_threshold()) else -(-m // quant.MAX_GEMV_TOKENS)
        total = 0
        for name, src, t, out_dim, in_dim, raw in self.weights.entries:
            total += groups * raw.size + 4 * m * (in_dim + out_dim)
        return total

    def close(self):
        for b in self._buffers:
            b.close()
        self._buffers = []
