"""Timed cases: layers of the five designs on prompts and on decoded tokens, at the sizes of the configurations in ``bench.py``.

A case is one pass of a layer module as a model calls it, with the step's metadata in the context: a whole decoder layer of
Qwen3, and the mixers and experts of the other designs behind their input projection.  Prompt steps run eagerly and decode steps
replay a captured graph, as the model runner does.  Sequences have unequal lengths and their pages are scattered.

Keys of a case: ``kind`` (which layer), ``step`` ('prompt' or 'decode'), ``width`` (1024 or 4096: the two sizes of every design),
``seqs`` and ``tokens`` (sequences and the longest one's tokens: brought in a prompt step, held in a decode step), ``before``
(tokens of a prompt that earlier portions or the prefix cache hold already), ``singles`` (decoding sequences that share the
step with the prompts) and ``option`` (one of the kind's ``OPTIONS``).
"""
import math
import random
from types import SimpleNamespace

import numpy as np
import torch

from tinyllmforge_amd.config import NO_WINDOW, ModelConfig
from tinyllmforge_amd.engine.inputs import decode_inputs, portion_inputs, portion_kind, prefill_inputs
from tinyllmforge_amd.layers.gla import GatedLinearAttention
from tinyllmforge_amd.layers.latent_attention import LatentAttention
from tinyllmforge_amd.layers.layernorm import RMSNorm
from tinyllmforge_amd.layers.moe import SwiGLUExperts
from tinyllmforge_amd.layers.pooled_attention import PooledWindowAttention
from tinyllmforge_amd.layers.residual_norm import ResidualLayerNorm
from tinyllmforge_amd.layers.rotary_embedding import rotation_table
from tinyllmforge_amd.layers.sink_attention import SinkAttention, query_temperatures
from tinyllmforge_amd.layers.ssd import StateSpace
from tinyllmforge_amd.layers.talking_attention import TalkingHeadsAttention
from tinyllmforge_amd.models.qwen3 import Qwen3DecoderLayer
from tinyllmforge_amd.utils.context import reset_context, set_context, set_portions_context

BF16, F32, F64 = torch.bfloat16, torch.float32, torch.float64
DEV = "cuda"
EPS = 1e-6
MAX_LEN = 8192 + 4096
YARN = dict(factor=8.0, original=4096, fast=16.0, slow=2.0)

# width -> query heads, KV heads, head dim, feed-forward
HEADS = {1024: (16, 8, 128, 3072), 4096: (32, 8, 128, 12288)}
# gated linear attention: heads, key dim, value dim
GLA = {1024: (8, 64, 128), 4096: (16, 128, 256)}
# latent attention: heads, dim, rotated dim, value dim, latent
LATENT = {1024: (16, 64, 32, 64, 256), 4096: (32, 128, 64, 128, 512)}
# experts, identity experts, top, feed-forward of an expert
EXPERTS = {1024: (32, 2, 4, 768), 4096: (64, 4, 8, 1536)}
# state-space layer: heads, value dim, state, groups
STATES = {1024: (32, 64, 128, 1), 4096: (128, 64, 128, 8)}


def listed():
    def case(name, kind, step, width, seqs, tokens, option="", before=0, singles=0):
        return dict(name=name, kind=kind, step=step, width=width, seqs=seqs, tokens=tokens, before=before, singles=singles, option=option)

    return [
        # one user talking to an 8B-size Qwen3 with int8 weights: the smallest call, launches and latency
        case("qwen3_decode_1", "qwen3", "decode", 4096, 1, 700, "w8a16"),
        # the same model serving a batch
        case("qwen3_decode_128", "qwen3", "decode", 4096, 128, 1100, "w8a16"),
        # a full prefill step of that batch: prompts of up to a thousand tokens
        case("qwen3_prompt_16x1024", "qwen3", "prompt", 4096, 16, 1024, "w8a16"),
        # prompts of the Gitopel design, its two mixers
        case("pooled_prompt_8x2048", "pooled", "prompt", 4096, 8, 2048),
        case("gla_prompt_8x2048", "gla", "prompt", 4096, 8, 2048),
        # prompts of Gigopel: windowed latent attention
        case("latent_prompt_8x2048", "latent", "prompt", 1024, 8, 2048, "window"),
        # prompts of Zuzunex with the convolution, and its experts under a middling batch of prompt rows
        case("sink_prompt_8x2048", "sink", "prompt", 4096, 8, 2048, "conv"),
        case("experts_rows_1021", "experts", "prompt", 1024, 1, 1021),
        # prompts of Tibenex: heads that mix their weights, state space; the latter as portions beside decoding sequences
        case("talk_prompt_8x2048", "talk", "prompt", 1024, 8, 2048),
        case("ssd_prompt_4x3000_mixed", "ssd", "prompt", 4096, 4, 3000, singles=33),
        # decoding: attention with long contexts, and a recurrence
        case("sink_decode_64", "sink", "decode", 1024, 64, 4096, "cap"),
        case("gla_decode_200", "gla", "decode", 1024, 200, 1500),
    ]


def draw(rng):
    spread = lambda lo, hi: round(math.exp(rng.uniform(math.log(lo), math.log(hi))))
    kind = rng.choice(sorted(KINDS))
    case = dict(kind=kind, step=rng.choice(["prompt", "prompt", "decode"]), width=rng.choice(sorted(HEADS)), before=0, singles=0,
                option=rng.choice(KINDS[kind].OPTIONS))
    if case["step"] == "decode":
        return case | dict(seqs=spread(1, 256), tokens=spread(16, 4096))
    rows = spread(24, 12000)
    tokens = min(rows, spread(24, 8192))
    case |= dict(seqs=min(256, max(1, rows // tokens)), tokens=tokens)
    if kind == "experts":
        return case
    if rng.random() < 0.3:
        block = KINDS[kind].BLOCK
        case["before"] = block * -(-spread(32, 2048) // block)
    if kind != "qwen3" and rng.random() < 0.3:
        case["singles"] = spread(1, 64)
    return case


# ------------------------------------------------------------------ a step's sequences
class Step:
    """The sequences of a case: ``lens[s]`` tokens brought on top of ``starts[s]`` held ones, singles first; ``tables[s]`` the pages
    and ``slots(s)`` the cache rows of everything a sequence holds after the step."""

    def __init__(self, case, block, long_portion=None):
        lengths = random.Random(f"{case['seqs']} {case['tokens']}")
        pages = random.Random(f"{case['tokens']} {case['seqs']}")
        longest, seqs = case["tokens"], case["seqs"]
        some = lambda lo: [longest] + [lengths.randint(max(1, longest // lo), longest) for _ in range(seqs - 1)]
        if case["step"] == "decode":
            pairs = [(1, n - 1) for n in some(8)]
        else:
            pairs = [(1, lengths.randint(1, 2048)) for _ in range(case["singles"])]
            pairs += sorted(((n, case["before"]) for n in some(2)), key=lambda p: portion_kind(p[0], long_portion))
        self.lens, self.starts = [p[0] for p in pairs], [p[1] for p in pairs]
        need = [-(-(n + s) // block) for n, s in pairs]
        self.block, self.pages = block, sum(need) + 2
        free = list(range(self.pages))
        pages.shuffle(free)
        self.tables = [[free.pop() for _ in range(k)] for k in need]
        self.rows = sum(self.lens)
        self.first = np.concatenate([[0], np.cumsum(self.lens)]).tolist()

    def sequences(self):
        """As the engine's input builders read them."""
        held = zip(self.lens, self.starts, self.tables)
        return [Sized(num_scheduled=n, num_computed=s, num_cached_tokens=s, num_cached_blocks=s // self.block, token_ids=range(n + s),
                      last_token=0, block_table=t, state_slot=i, size=n + s) for i, (n, s, t) in enumerate(held)]

    def slots(self, s):
        at = torch.arange(self.starts[s] + self.lens[s], device=DEV)
        return torch.tensor(self.tables[s], device=DEV)[at // self.block] * self.block + at % self.block

    def new_rows(self, s):
        return slice(self.first[s], self.first[s + 1])

    def positions(self, s):
        return torch.arange(self.starts[s], self.starts[s] + self.lens[s], device=DEV)

    def keys_seen(self, window=1 << 30, pool=None):
        """Key rows that the step's rows attend to, all together."""
        total = 0
        for n, s in zip(self.lens, self.starts):
            at = np.arange(s, s + n, dtype=np.int64) + 1
            total += int(np.minimum(at, window).sum())
            if pool:
                total += int((np.maximum(at - window, 0) // pool).sum())
        return total

    def keys_held(self, window=1 << 30):
        """Cache rows that some row of the step attends to."""
        return sum(min(n + s, n - 1 + window) for n, s in zip(self.lens, self.starts))


class Sized(SimpleNamespace):
    def __len__(self):
        return self.size


def on_gpu(arrays):
    return {k: torch.from_numpy(v).to(DEV) if isinstance(v, np.ndarray) else v for k, v in arrays.items()}


# ------------------------------------------------------------------ 64-bit arithmetic of the kinds
def rms(x, eps=EPS):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def silu(z):
    return z * torch.sigmoid(z)


def frequencies(dims, base, factor=None, original=None, fast=None, slow=None):
    f = base ** (-torch.arange(0, dims, 2, dtype=F64, device=DEV) / dims)
    if factor is None:
        return f, 1.0
    pair = lambda turns: dims * math.log(original / (2 * math.pi * turns)) / (2 * math.log(base))
    lo, hi = max(math.floor(pair(fast)), 0), min(math.ceil(pair(slow)), dims - 1)
    ramp = ((torch.arange(dims // 2, dtype=F64, device=DEV) - lo) / max(hi - lo, 0.001)).clamp(0, 1)
    return f / factor * ramp + f * (1 - ramp), 0.1 * math.log(factor) + 1


def rotated(x, positions, halves, dims, base, **scaling):
    """``x [T, H, D]``, the first ``dims`` dimensions."""
    f, mult = frequencies(dims, base, **scaling)
    a = positions.to(F64)[:, None, None] * f
    c, s = a.cos() * mult, a.sin() * mult
    out = x.clone()
    at = (slice(0, dims // 2), slice(dims // 2, dims)) if halves else (slice(0, dims, 2), slice(1, dims, 2))
    u, v = x[..., at[0]], x[..., at[1]]
    out[..., at[0]], out[..., at[1]] = u * c - v * s, v * c + u * s
    return out


def weights_of(scores, positions, window=1 << 30, sink=None):
    """Softmax over the last dimension (keys from position 0 on) of what a row at ``positions`` sees."""
    keys = torch.arange(scores.shape[-1], device=DEV)
    hidden = (keys > positions[:, None]) | (keys <= positions[:, None] - window)
    scores = scores.masked_fill(hidden, -math.inf)
    top = scores.amax(-1, keepdim=True)
    if sink is not None:
        top = top.clamp(min=float(sink))
    e = torch.exp(scores - top)
    return e / (e.sum(-1, keepdim=True) + (torch.exp(sink - top) if sink is not None else 0))


def causal_conv(new, earlier, taps):
    """``new [T, C]`` after the ``taps - 1`` rows ``earlier``; ``taps [n, C]``, the last one meets the row itself."""
    u = torch.cat([earlier, new])
    return sum(taps[j] * u[j:j + new.shape[0]] for j in range(taps.shape[0]))


def ring_rows(ring, start, channels):
    """The rows before position ``start`` of a ring (position p in row p mod taps), zeros below position 0."""
    taps = ring.shape[0]
    rows = [ring[p % taps] if p >= 0 else torch.zeros(channels, dtype=F64, device=DEV) for p in range(start - taps + 1, start)]
    return torch.stack([r.to(F64) for r in rows])


def kept_ring(ring, start, new):
    """``ring`` with the rows that the next token needs of ``new`` (positions from ``start`` on) in their places."""
    taps, out = ring.shape[0], ring.to(F64).clone()
    for i in range(max(0, new.shape[0] - taps + 1), new.shape[0]):
        out[(start + i) % taps] = new[i]
    return out


def rows_at(n, size=1024):
    return [slice(i, min(n, i + size)) for i in range(0, n, size)]


def padded(rows, lens):
    """``[T, ...]`` of each sequence -> ``[longest, sequences, ...]`` with zeros."""
    out = torch.zeros(max(lens), len(lens), *rows[0].shape[1:], dtype=F64, device=DEV)
    for i, r in enumerate(rows):
        out[:len(r), i] = r
    return out


# ------------------------------------------------------------------ the kinds
class Kind:
    """``data(case, seed)``: inputs, weights and caches; ``layer(d)``: the module with them; ``call(layer, d)``: one pass;
    ``exact(d)``: its outputs in 64 bits."""
    OPTIONS, BLOCK, LONG, WINDOWS = [""], 64, None, ()

    def __init__(self, case, seed=None):
        self.case, self.width = case, case["width"]
        self.sizes()
        self.step = Step(case, self.BLOCK, self.LONG)
        if seed is not None:
            self.gen = torch.Generator(device=DEV).manual_seed(seed)
            self.data()

    def randn(self, *shape, dtype=BF16, scale=1.0, mean=0.0):
        out = torch.empty(shape, dtype=F32 if dtype == F32 else BF16, device=DEV).normal_(mean, scale, generator=self.gen)
        return out if dtype == out.dtype else out.to(dtype)

    def metadata(self):
        arrays = portion_inputs(self.step.sequences(), self.BLOCK, self.LONG, self.windows())
        d = on_gpu(arrays)
        self.positions = d.pop("positions")
        d.pop("input_ids")
        self.fields = dict(d, max_len=MAX_LEN)

    def windows(self):
        return ()

    def publish(self):
        set_portions_context(**self.fields)

    def held(self, cache, s):
        """Rows of sequence ``s`` before the step, of a cache ``[pages, block, ...]``."""
        return cache.flatten(0, 1)[self.step.slots(s)[:self.step.starts[s]]].to(F64)

    def scatter(self, cache, s, rows):
        """In place, on a cache ``[pages, block, ...]`` in 64 bits: the step's rows of sequence ``s``."""
        flat = cache.flatten(0, 1)
        flat[self.step.slots(s)[self.step.starts[s]:], ..., :rows.shape[-1]] = rows

    def tolerance(self):
        """About four times what the outputs are off from 64 bits: bf16 inputs of the products and bf16 results."""
        return {"rel": 1.3e-2, "max": 0.2}


class Qwen3(Kind):
    """A decoder layer of Qwen3 from after its input norm to after the next one; ``option``: int8 or bf16 weights, e4m3 cache."""
    OPTIONS, BLOCK = ["w8a16", "bf16", "w8a16 fp8"], 256

    def sizes(self):
        self.hq, self.hkv, self.dim, self.ff = HEADS[self.width]
        self.int8, self.fp8 = "w8a16" in self.case["option"], "fp8" in self.case["option"]
        self.shapes = dict(qkv=((self.hq + 2 * self.hkv) * self.dim, self.width), o=(self.width, self.hq * self.dim),
                           gate_up=(2 * self.ff, self.width), down=(self.width, self.ff))

    def data(self):
        w, n = self.width, self.step.rows
        self.weights = {}
        for name, (rows, cols) in self.shapes.items():
            if self.int8:
                q = torch.randint(-127, 128, (rows, cols), dtype=torch.int8, device=DEV, generator=self.gen)
                scale = torch.rand(rows, device=DEV, generator=self.gen) * 0.5 + 0.75
                self.weights[name] = q, scale / 73 * cols ** -0.5
            else:
                self.weights[name] = self.randn(rows, cols, scale=cols ** -0.5), None
        self.norms = {k: self.randn(s, scale=0.1, mean=1.0) for k, s in (("q", self.dim), ("k", self.dim), ("post", w), ("next", w))}
        cache = (self.step.pages, self.BLOCK, self.hkv, self.dim)
        self.k, self.v = self.randn(*cache), self.randn(*cache)
        if self.fp8:
            self.scale = torch.full((self.hkv,), 1 / 16, device=DEV)
            self.k, self.v = ((t.float() * 16).to(torch.float8_e4m3fn) for t in (self.k, self.v))
        self.normed, self.residual = self.randn(n, w), self.randn(n, w)

    def layer(self):
        cfg = ModelConfig(hidden_size=self.width, num_hidden_layers=1, num_attention_heads=self.hq, num_key_value_heads=self.hkv,
                          intermediate_size=self.ff, vocab_size=16, head_dim=self.dim, max_position_embeddings=MAX_LEN)
        layer = built(Qwen3DecoderLayer, cfg)
        attn, mlp = layer.self_attn, layer.mlp
        for lin, name in ((attn.qkv_proj, "qkv"), (attn.o_proj, "o"), (mlp.gate_up_proj, "gate_up"), (mlp.down_proj, "down")):
            w, scale = self.weights[name]
            if self.int8:
                lin.load_quantized(w, scale)
                lin.finish_quantized_load()
                lin.pack_()
            else:
                lin.weight.data.copy_(w)
                if name == "gate_up":
                    lin.interleave_()
        self.next = built(RMSNorm, self.width, EPS)
        for norm, name in ((attn.q_norm, "q"), (attn.k_norm, "k"), (layer.post_attention_layernorm, "post"), (self.next, "next")):
            norm.weight.data.copy_(self.norms[name])
        attn.attn.k_cache, attn.attn.v_cache = self.k, self.v
        if self.fp8:
            attn.attn.k_scale = attn.attn.v_scale = self.scale
        return layer

    def metadata(self):
        seqs = self.step.sequences()
        if self.case["step"] == "decode":
            d = on_gpu(decode_inputs(seqs, self.BLOCK, position_quirk=False))
            self.fields = dict(is_prefill=False, slot_mapping=d["slot_mapping"], context_lens=d["context_lens"], block_tables=d["block_tables"])
        else:
            d = on_gpu(prefill_inputs(seqs, self.BLOCK))
            self.fields = dict(is_prefill=True, **{k: d[k] for k in ("cu_seqlens_q", "cu_seqlens_k", "max_seqlen_q", "max_seqlen_k",
                                                                     "slot_mapping", "block_tables")})
        self.positions = d["positions"]

    def publish(self):
        set_context(**self.fields)

    def call(self, layer):
        normed, residual = layer.forward_normed(self.positions, self.normed, self.residual, self.next)
        return {"normed": normed, "residual": residual, "k": self.k, "v": self.v}

    def exact(self):
        def linear(x, name):
            w, scale = self.weights[name]
            y = torch.cat([x @ part.to(F64).T for part in w.split(4096)], dim=1)
            return y * scale.to(F64) if scale is not None else y

        n, norms = self.step.rows, {k: v.to(F64) for k, v in self.norms.items()}
        q, k, v = linear(self.normed.to(F64), "qkv").view(n, -1, self.dim).split([self.hq, self.hkv, self.hkv], dim=1)
        positions = torch.cat([self.step.positions(s) for s in range(len(self.step.lens))])
        rope = dict(halves=True, dims=self.dim, base=1e6)
        q, k = rotated(rms(q) * norms["q"], positions, **rope), rotated(rms(k) * norms["k"], positions, **rope)
        o, caches = torch.empty(n, self.hq, self.dim, dtype=F64, device=DEV), [self.k.to(F64), self.v.to(F64)]
        mult = 1 / 16 if self.fp8 else 1
        for s, at in ((s, self.step.new_rows(s)) for s in range(len(self.step.lens))):
            ks, vs = (torch.cat([self.held(c, s) * mult, t[at]]) for c, t in zip((self.k, self.v), (k, v)))
            for h in range(self.hq):
                scores = q[at, h] @ ks[:, h * self.hkv // self.hq].T * self.dim ** -0.5
                o[at, h] = weights_of(scores, self.step.positions(s)) @ vs[:, h * self.hkv // self.hq]
            for cache, t in zip(caches, (k, v)):
                self.scatter(cache, s, t[at] / mult)
        x = self.residual.to(F64) + linear(o.view(n, -1), "o")
        gate, up = linear(rms(x) * norms["post"], "gate_up").split(self.ff, dim=1)
        x = x + linear(silu(gate) * up, "down")
        k, v = caches if not self.fp8 else (None, None)
        return {"normed": rms(x) * norms["next"], "residual": x, "k": k, "v": v}

    def work(self):
        n, item = self.step.rows, 1 if self.fp8 else 2
        weights = sum(a * b for a, b in self.shapes.values())
        kv = self.step.keys_held() * 2 * self.hkv * self.dim * item
        return {"bytes": weights * (1 if self.int8 else 2) + kv + n * self.width * 8,
                "flops": 2.0 * n * weights + 4.0 * self.hq * self.dim * self.step.keys_seen()}

    def tolerance(self):
        # an e4m3 value on the border of two codes may become either
        return {"rel": 4e-2 if self.fp8 else 1.6e-2, "max": 0.9 if self.fp8 else 0.3}


class Pooled(Kind):
    """Gitopel's attention: sigmoid weights over a window of 1024 and the means of the blocks of 16 behind it."""
    WINDOW, POOL = 1024, 16

    def sizes(self):
        self.h, self.g, self.d, _ = HEADS[self.width]

    def data(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        self.proj = self.randn(n, -(-((h + g) * d + h) // 16) * 16)
        self.qb, self.kb, self.bias = self.randn(h * d, scale=0.1), self.randn(g * d, scale=0.1), self.randn(h, scale=0.3, mean=-5.0)
        self.k, self.v = self.randn(self.step.pages, self.BLOCK, g, d), self.randn(self.step.pages, self.BLOCK, g, d)
        self.k.copy_(rms(self.k.float()))
        mean = lambda t: t.float().view(self.step.pages, -1, self.POOL, g, d).mean(2).to(BF16)
        self.pk, self.pv = mean(self.k), mean(self.v)

    def layer(self):
        rope = rotation_table(self.d, MAX_LEN, 1e4).to(DEV)
        layer = built(PooledWindowAttention, self.h, self.g, self.d, self.d ** -0.5, self.WINDOW, self.POOL, self.d, rope, EPS, BF16)
        layer.score_bias.data.copy_(self.bias)
        layer.bind_pages(self.step.pages, self.BLOCK, DEV)
        for name in ("k", "v", "pk", "pv"):
            getattr(layer.kv, name).copy_(getattr(self, name))
        return layer

    def call(self, layer):
        out = layer(self.proj, self.qb, self.kb, self.positions)
        return {"out": out, "k": layer.kv.k, "v": layer.kv.v}

    def exact(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        q, k, gate = self.proj.to(F64)[:, :(h + g) * d + h].split([h * d, g * d, h], dim=1)
        q, k = (q + self.qb.to(F64)).view(n, h, d), (k + self.kb.to(F64)).view(n, g, d)
        out, caches = torch.empty(n, h, d, dtype=F64, device=DEV), [self.k.to(F64), self.v.to(F64)]
        for s, at in ((s, self.step.new_rows(s)) for s in range(len(self.step.lens))):
            pos = self.step.positions(s)
            qs, ks = (rms(rotated(t[at], pos, False, d, 1e4)) for t in (q, k))
            self.scatter(caches[0], s, ks)
            self.scatter(caches[1], s, k[at])
            ks, vs = torch.cat([self.held(self.k, s), ks]), torch.cat([self.held(self.v, s), k[at]])
            blocks = len(ks) // self.POOL
            pk, pv = (t[:blocks * self.POOL].view(blocks, self.POOL, g, d).mean(1) for t in (ks, vs))
            keys, ends = torch.arange(len(ks), device=DEV), torch.arange(blocks, device=DEV) * self.POOL + self.POOL - 1
            seen = torch.cat([(keys <= pos[:, None]) & (keys > pos[:, None] - self.WINDOW), ends <= pos[:, None] - self.WINDOW], dim=1)
            for i in range(h):
                kv = i * g // h
                scores = qs[:, i] @ torch.cat([ks[:, kv], pk[:, kv]]).T * d ** -0.5 + self.bias[i].to(F64)
                out[at, i] = (torch.sigmoid(scores) * seen) @ torch.cat([vs[:, kv], pv[:, kv]])
        out = out * torch.sigmoid(gate)[:, :, None]
        return {"out": out.view(n, -1), "k": caches[0], "v": caches[1]}

    def work(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        seen, held = self.step.keys_seen(self.WINDOW, self.POOL), self.step.keys_held(self.WINDOW)
        return {"bytes": 2.0 * (n * ((h + g) * d + h + h * d) + held * 2 * g * d), "flops": 4.0 * h * d * seen}

    def tolerance(self):
        return {"rel": 1.7e-2, "max": 0.3}


class Gla(Kind):
    """Gitopel's gated linear attention: a decay per key channel, an fp32 state."""
    RANK, TAU = 16, 16.0

    def sizes(self):
        self.h, self.dk, self.dv = GLA[self.width]

    def data(self):
        n, h, dk, dv = self.step.rows, self.h, self.dk, self.dv
        self.proj = self.randn(n, -(-(2 * h * (dk + dv) + self.RANK) // 16) * 16)
        self.a2, self.a2b = self.randn(h * dk, self.RANK, scale=0.3), self.randn(h * dk, scale=0.5, mean=1.0)
        self.norm = self.randn(dv, scale=0.1, mean=1.0)
        self.state = self.randn(len(self.step.lens), h, dk, dv, dtype=F32, scale=3.0)

    def layer(self):
        layer = built(GatedLinearAttention, self.h, self.dk, self.dv, self.RANK, self.TAU, EPS)
        for p, t in ((layer.decay_weight, self.a2), (layer.decay_bias, self.a2b), (layer.norm.weight, self.norm)):
            p.data.copy_(t)
        layer.bind_slots(len(self.step.lens), DEV)
        layer.state.copy_(self.state)
        return layer

    def call(self, layer):
        return {"out": layer(self.proj, self.positions), "state": layer.state}

    def exact(self):
        n, h, dk, dv, lens = self.step.rows, self.h, self.dk, self.dv, self.step.lens
        x = self.proj.to(F64)[:, :2 * h * (dk + dv) + self.RANK]
        q, k, v, g, r = x.split([h * dk, h * dk, h * dv, h * dv, self.RANK], dim=1)
        decay = -torch.nn.functional.softplus(-(r @ self.a2.to(F64).T + self.a2b.to(F64))) / self.TAU
        q, k, decay, v = (padded([t[self.step.new_rows(s)].view(lens[s], h, -1) for s in range(len(lens))], lens)
                          for t in (q * dk ** -0.5, k, decay, v))
        state = self.state.to(F64) * (torch.tensor(self.step.starts, device=DEV) > 0)[:, None, None, None]
        out = torch.empty_like(v)
        for t in range(max(lens)):
            state = state * decay[t, ..., None].exp() + k[t, ..., None] * v[t, :, :, None]
            out[t] = (state * q[t, ..., None]).sum(2)
        o = torch.cat([out[:m, s] for s, m in enumerate(lens)])
        o = (rms(o) * self.norm.to(F64)).reshape(n, -1)
        return {"out": o * silu(g), "state": state}

    def work(self):
        n, h, dk, dv = self.step.rows, self.h, self.dk, self.dv
        states = sum(1 + (s > 0) for s in self.step.starts)
        return {"bytes": 2.0 * n * (2 * h * (dk + dv) + self.RANK + h * dv) + 4.0 * states * h * dk * dv, "flops": 4.0 * n * h * dk * dv}

    def tolerance(self):
        return {"rel": 7e-3, "max": 0.1}


class Latent(Kind):
    """Gigopel's latent attention behind its projection; ``option``: a window of 1024 or none."""
    OPTIONS, LONG = ["window", "causal"], 128

    def sizes(self):
        self.h, self.d, self.r, self.vd, self.rank = LATENT[self.width]
        self.window = 1024 if self.case["option"] == "window" else NO_WINDOW

    def windows(self):
        return (self.window,)

    def data(self):
        n, h, d, r, vd, rank = self.step.rows, self.h, self.d, self.r, self.vd, self.rank
        self.proj = self.randn(n, h * (d + r) + rank + r)
        self.norm = self.randn(rank, scale=0.1, mean=1.0)
        self.uk, self.uv = self.randn(h * d, rank, scale=rank ** -0.5), self.randn(h * vd, rank, scale=rank ** -0.5)
        self.cache = self.randn(self.step.pages, self.BLOCK, rank + r)

    def layer(self):
        h, d, r, vd, rank = self.h, self.d, self.r, self.vd, self.rank
        layer = built(LatentAttention, h, d, r, rank, vd, (d + r) ** -0.5, self.window, 0, rotation_table(r, MAX_LEN, 1e4).to(DEV), EPS, BF16)
        for p, t in ((layer.norm.weight, self.norm), (layer.uk, self.uk), (layer.uv, self.uv)):
            p.data.copy_(t)
        layer.pack_()
        layer.bind_pages(self.step.pages, self.BLOCK, DEV)
        layer.cache[..., :rank + r].copy_(self.cache)
        return layer

    def call(self, layer):
        q = layer.prepare(self.proj, self.h * (self.d + self.r), self.positions)
        out = torch.empty(q.shape[0], self.h * self.vd, dtype=BF16, device=DEV)
        layer(q, self.positions, out)
        return {"out": out, "cache": layer.cache}

    def exact(self):
        n, h, d, r, vd, rank = self.step.rows, self.h, self.d, self.r, self.vd, self.rank
        q, c, kr = self.proj.to(F64).split([h * (d + r), rank, r], dim=1)
        q, c = q.view(n, h, d + r), rms(c) * self.norm.to(F64)
        cache = torch.zeros(self.step.pages, self.BLOCK, -(-(rank + r) // 64) * 64, dtype=F64, device=DEV)
        cache[..., :rank + r] = self.cache
        out = torch.empty(n, h, vd, dtype=F64, device=DEV)
        uk, uv = self.uk.to(F64).view(h, d, rank), self.uv.to(F64).view(h, vd, rank)
        for s, at in ((s, self.step.new_rows(s)) for s in range(len(self.step.lens))):
            pos = self.step.positions(s)
            rows = torch.cat([c[at], rotated(kr[at][:, None], pos, False, r, 1e4)[:, 0]], dim=1)
            self.scatter(cache, s, rows)
            rows = torch.cat([self.held(self.cache, s), rows])
            turned = rotated(q[at][..., d:].contiguous(), pos, False, r, 1e4)
            for i in range(h):
                scores = (q[at, i, :d] @ (rows[:, :rank] @ uk[i].T).T + turned[:, i] @ rows[:, rank:].T) * (d + r) ** -0.5
                out[at, i] = weights_of(scores, pos, self.window) @ (rows[:, :rank] @ uv[i].T)
        return {"out": out.view(n, -1), "cache": cache}

    def work(self):
        n, h, d, r, vd, rank = self.step.rows, self.h, self.d, self.r, self.vd, self.rank
        held, seen = self.step.keys_held(self.window), self.step.keys_seen(self.window)
        return {"bytes": 2.0 * (n * (h * (d + r) + rank + r + h * vd) + held * (rank + r) + h * (d + vd) * rank),
                "flops": 2.0 * h * (d + r + vd) * seen + 2.0 * n * h * (d + vd) * rank}


class Sink(Kind):
    """Zuzunex's attention: capped scores with temperatures, or ('conv') biases, a short convolution and rotation."""
    OPTIONS, LONG, TAPS = ["cap", "conv"], 16, 4

    def sizes(self):
        self.h, self.g, self.d, _ = HEADS[self.width]
        self.conv, self.channels = self.case["option"] == "conv", (self.h + 2 * self.g) * self.d

    def data(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        self.proj, self.sink = self.randn(n, self.channels + h * d), self.randn(h)
        if self.conv:
            self.bias, self.taps = self.randn(self.channels, scale=0.1), self.randn(self.TAPS, self.channels, scale=0.5)
            self.qn, self.kn = self.randn(d, scale=0.1, mean=1.0), self.randn(d, scale=0.1, mean=1.0)
            self.ring = self.randn(len(self.step.lens), self.TAPS, self.channels)
        self.k, self.v = self.randn(self.step.pages, g, self.BLOCK, d), self.randn(self.step.pages, g, self.BLOCK, d)

    def layer(self):
        extra = dict(bias=True, taps=self.TAPS, weighted_norm=True, rot_dims=self.d, rope=rotation_table(self.d, MAX_LEN, 1e6, **YARN).to(DEV)) \
            if self.conv else dict(cap=20.0, temperatures=query_temperatures(0.1, 1024, MAX_LEN).to(DEV))
        layer = built(SinkAttention, self.h, self.g, self.d, self.d, self.d ** -0.5, EPS, BF16, **extra)
        layer.sink.data.copy_(self.sink)
        layer.bind_pages(self.step.pages, self.BLOCK, DEV)
        layer.bind_slots(len(self.step.lens), DEV)
        layer.kv[0].k.copy_(self.k)
        layer.kv[0].v.copy_(self.v)
        if self.conv:
            for p, t in ((layer.bias, self.bias), (layer.conv, self.taps), (layer.q_norm.weight, self.qn), (layer.k_norm.weight, self.kn)):
                p.data.copy_(t)
            layer.rings[0].copy_(self.ring)
        return layer

    def call(self, layer):
        out = {"out": layer(self.proj, self.positions), "k": layer.kv[0].k, "v": layer.kv[0].v}
        return out | ({"ring": layer.rings[0]} if self.conv else {})

    def exact(self):
        n, h, g, d, channels = self.step.rows, self.h, self.g, self.d, self.channels
        x, gate = self.proj.to(F64).split([channels, h * d], dim=1)
        out = torch.empty(n, h, d, dtype=F64, device=DEV)
        caches = [t.to(F64).transpose(1, 2).contiguous() for t in (self.k, self.v)]
        rings = []
        for s, at in ((s, self.step.new_rows(s)) for s in range(len(self.step.lens))):
            pos, start, u = self.step.positions(s), self.step.starts[s], x[at]
            if self.conv:
                rings.append(kept_ring(self.ring[s], start, u))
                bias, earlier = self.bias.to(F64), ring_rows(self.ring[s], start, channels)
                real = torch.tensor([p >= 0 for p in range(start - self.TAPS + 1, start)], device=DEV)[:, None]
                u = causal_conv(u + bias, (earlier + bias) * real, self.taps.to(F64))
            q, k, v = u.view(len(u), -1, d).split([h, g, g], dim=1)
            q, k = rms(q), rms(k)
            if self.conv:
                q, k = (rotated(t * w.to(F64), pos, True, d, 1e6, **YARN) for t, w in ((q, self.qn), (k, self.kn)))
            else:
                q = q * (1 + 0.1 * torch.log(((pos + 1) // 1024 + 1).to(F64)))[:, None, None]
            ks, vs = (torch.cat([self.held(c, s), t]) for c, t in zip(caches, (k, v)))
            for c, t in zip(caches, (k, v)):
                self.scatter(c, s, t)
            for i in range(h):
                scores = q[:, i] @ ks[:, i * g // h].T * d ** -0.5
                scores = scores if self.conv else 20 * torch.tanh(scores / 20)
                out[at, i] = weights_of(scores, pos, sink=self.sink[i].to(F64)) @ vs[:, i * g // h]
        result = {"out": out.view(n, -1) * torch.sigmoid(gate), "k": caches[0].transpose(1, 2), "v": caches[1].transpose(1, 2)}
        return result | ({"ring": torch.stack(rings)} if self.conv else {})

    def work(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        return {"bytes": 2.0 * (n * (self.channels + 2 * h * d) + self.step.keys_held() * 2 * g * d),
                "flops": 4.0 * h * d * self.step.keys_seen()}


class Talk(Kind):
    """Tibenex's attention whose heads mix their weights."""
    LONG = 128

    def sizes(self):
        self.h, self.g, self.d, _ = HEADS[self.width]

    def data(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        self.proj = self.randn(n, (h + 2 * g) * d)
        self.qn, self.kn, self.temp = (self.randn(s, scale=0.1, mean=1.0) for s in (h * d, g * d, h))
        self.talk = (torch.eye(h, device=DEV) + self.randn(h, h, scale=0.2)).to(BF16)
        self.k, self.v = self.randn(self.step.pages, g, self.BLOCK, d), self.randn(self.step.pages, g, self.BLOCK, d)

    def layer(self):
        layer = built(TalkingHeadsAttention, self.h, self.g, self.d, self.d, self.d ** -0.5, EPS, BF16, self.d,
                      rotation_table(self.d, MAX_LEN, 1e6).to(DEV))
        for p, t in ((layer.q_norm.weight, self.qn), (layer.k_norm.weight, self.kn), (layer.temp, self.temp), (layer.talk, self.talk)):
            p.data.copy_(t)
        layer.bind_pages(self.step.pages, self.BLOCK, DEV)
        layer.kv.k.copy_(self.k)
        layer.kv.v.copy_(self.v)
        return layer

    def call(self, layer):
        return {"out": layer(self.proj, self.positions), "k": layer.kv.k, "v": layer.kv.v}

    def exact(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        q, k, v = self.proj.to(F64).split([h * d, g * d, g * d], dim=1)
        q, k, v = (rms(q) * self.qn.to(F64)).view(n, h, d), (rms(k) * self.kn.to(F64)).view(n, g, d), v.view(n, g, d)
        out = torch.empty(n, h, d, dtype=F64, device=DEV)
        caches = [t.to(F64).transpose(1, 2).contiguous() for t in (self.k, self.v)]
        talk = self.talk.to(F64)
        for s, at in ((s, self.step.new_rows(s)) for s in range(len(self.step.lens))):
            pos = self.step.positions(s)
            qs, kn = (rotated(t[at], pos, False, d, 1e6) for t in (q, k))
            ks, vs = (torch.cat([self.held(c, s), t]) for c, t in zip(caches, (kn, v[at])))
            for c, t in zip(caches, (kn, v[at])):
                self.scatter(c, s, t)
            for part in rows_at(len(pos), 512):
                w = torch.stack([weights_of(qs[part, i] @ ks[:, i * g // h].T * (d ** -0.5 * self.temp[i].to(F64)), pos[part]) for i in range(h)])
                mixed = (talk @ w.view(h, -1)).view(w.shape)
                out[at.start + part.start:at.start + part.stop] = torch.stack([mixed[i] @ vs[:, i * g // h] for i in range(h)], dim=1)
        return {"out": out.view(n, -1), "k": caches[0].transpose(1, 2), "v": caches[1].transpose(1, 2)}

    def work(self):
        n, h, g, d = self.step.rows, self.h, self.g, self.d
        return {"bytes": 2.0 * (n * (2 * h + 2 * g) * d + self.step.keys_held() * 2 * g * d),
                "flops": (4.0 * h * d + 2.0 * h * h) * self.step.keys_seen()}


class Ssd(Kind):
    """Tibenex's state-space layer: convolution, fp32 state, gated norm in parts."""
    LONG, TAPS = 128, 4

    def sizes(self):
        self.h, self.p, self.n, self.g = STATES[self.width]
        self.inner = self.h * self.p
        self.channels = self.inner + 2 * self.g * self.n

    def data(self):
        seqs = len(self.step.lens)
        self.proj = self.randn(self.step.rows, -(-(self.inner + self.channels + self.h) // 16) * 16)
        self.conv, self.conv_bias = self.randn(self.TAPS, self.channels, scale=0.5), self.randn(self.channels, scale=0.1)
        self.dt_bias, self.a_log, self.dd = self.randn(self.h, scale=0.5, mean=-3.0), self.randn(self.h, scale=0.5, mean=1.0), self.randn(self.h)
        self.norm = self.randn(self.inner, scale=0.1, mean=1.0)
        self.state = self.randn(seqs, self.h, self.n, self.p, dtype=F32)
        self.ring = self.randn(seqs, self.TAPS, self.channels)

    def layer(self):
        layer = built(StateSpace, self.h, self.p, self.n, self.g, self.TAPS, self.g, EPS, BF16)
        for p, t in ((layer.conv, self.conv), (layer.conv_bias, self.conv_bias), (layer.dt_bias, self.dt_bias), (layer.A_log, self.a_log),
                     (layer.D, self.dd), (layer.norm.weight, self.norm)):
            p.data.copy_(t)
        layer.bind_slots(len(self.step.lens), DEV)
        layer.state.copy_(self.state)
        layer.ring.copy_(self.ring)
        return layer

    def call(self, layer):
        return {"out": layer(self.proj, self.positions), "state": layer.state, "ring": layer.ring}

    def exact(self):
        rows, lens, starts = self.step.rows, self.step.lens, self.step.starts
        h, p, n, g = self.h, self.p, self.n, self.g
        z, xbc, dt = self.proj.to(F64)[:, :self.inner + self.channels + h].split([self.inner, self.channels, h], dim=1)
        dt = torch.nn.functional.softplus(dt + self.dt_bias.to(F64))
        rings, parts = [], []
        for s in range(len(lens)):
            at = self.step.new_rows(s)
            rings.append(kept_ring(self.ring[s], starts[s], xbc[at]))
            u = causal_conv(xbc[at], ring_rows(self.ring[s], starts[s], self.channels), self.conv.to(F64)) + self.conv_bias.to(F64)
            parts.append(silu(u).split([self.inner, g * n, g * n], dim=1))
        x = padded([u[0].view(-1, h, p) for u in parts], lens)
        b, c = (padded([u[i].view(-1, g, n) for u in parts], lens) for i in (1, 2))
        dt = padded([dt[self.step.new_rows(s)] for s in range(len(lens))], lens)
        decay = torch.exp(-torch.exp(self.a_log.to(F64)) * dt)
        state = self.state.to(F64) * (torch.tensor(starts, device=DEV) > 0)[:, None, None, None]
        out, share = torch.empty_like(x), h // g
        for t in range(max(lens)):
            bt, ct = b[t].repeat_interleave(share, 1), c[t].repeat_interleave(share, 1)
            state = state * decay[t][..., None, None] + (bt * dt[t][..., None])[..., None] * x[t][:, :, None, :]
            out[t] = (state * ct[..., None]).sum(2)
        out = out + self.dd.to(F64)[:, None] * x
        y = torch.cat([out[:m, s] for s, m in enumerate(lens)]).reshape(rows, -1) * silu(z)
        y = rms(y.view(rows, g, -1)).reshape(rows, -1) * self.norm.to(F64)
        return {"out": y, "state": state, "ring": torch.stack(rings)}

    def work(self):
        rows, states = self.step.rows, sum(1 + (s > 0) for s in self.step.starts)
        return {"bytes": 2.0 * rows * (2 * self.inner + self.channels + self.h) + 4.0 * states * self.h * self.n * self.p,
                "flops": 4.0 * rows * self.h * self.n * self.p}


class Experts(Kind):
    """Zuzunex's mixture of experts with the residual add and layer norm that take its rows."""

    def sizes(self):
        self.experts, self.identity, self.top, self.ff = EXPERTS[self.width]

    def data(self):
        w, n, e = self.width, self.step.rows, self.experts
        self.hidden, self.x = self.randn(n, w), self.randn(n, w, dtype=F32)
        self.router, self.correction = self.randn(e + self.identity, w, scale=w ** -0.5), self.randn(e + self.identity, scale=0.01)
        self.gate, self.up = self.randn(e, self.ff, w, scale=w ** -0.5), self.randn(e, self.ff, w, scale=w ** -0.5)
        self.down = self.randn(e, w, self.ff, scale=self.ff ** -0.5)
        self.norm, self.norm_bias = self.randn(w, scale=0.1, mean=1.0), self.randn(w, scale=0.1)

    def layer(self):
        layer = built(SwiGLUExperts, self.width, self.experts, self.top, self.ff, self.identity)
        layer.weight_loader(layer.router, self.router, "router")
        layer.correction.data.copy_(self.correction)
        groups = layer.gate_up.data.view(self.experts, self.ff // 8, 2, 8, self.width)
        groups[:, :, 0].copy_(self.gate.view(self.experts, -1, 8, self.width))
        groups[:, :, 1].copy_(self.up.view(self.experts, -1, 8, self.width))
        layer.down.data[:, :self.width].copy_(self.down)
        layer.zero_pads_()
        self.after = built(ResidualLayerNorm, self.width, EPS)
        self.after.weight.data.copy_(self.norm)
        self.after.bias.data.copy_(self.norm_bias)
        return layer

    def call(self, layer):
        h = self.after.after_adding(None, self.x, *layer(self.hidden))
        return {"h": h, "x": self.x}

    def exact(self):
        h, e = self.hidden.to(F64), self.experts
        scores = torch.softmax(h @ self.router.to(F64).T, dim=1)
        chosen = (scores + self.correction.to(F64)).topk(self.top, dim=1).indices
        weights = scores.gather(1, chosen)
        weights = weights / (weights.sum(1, keepdim=True) + 1e-20)
        x = self.x.to(F64)
        for i in range(e + self.identity):
            at, k = (chosen == i).nonzero(as_tuple=True)
            rows = h[at]
            if i < e:
                gate, up, down = (t[i].to(F64) for t in (self.gate, self.up, self.down))
                rows = (silu(rows @ gate.T) * (rows @ up.T)) @ down.T
            x.index_add_(0, at, rows * weights[at, k][:, None])
        centred = x - x.mean(1, keepdim=True)
        out = rms(centred) * self.norm.to(F64) + self.norm_bias.to(F64)
        return {"h": out, "x": x}

    def work(self):
        n, w = self.step.rows, self.width
        share = self.experts / (self.experts + self.identity)
        rows = n * self.top * share
        touched = self.experts * (1 - (1 - 1 / self.experts) ** rows)
        return {"bytes": 2.0 * touched * 3 * self.ff * w + n * w * 12.0, "flops": 6.0 * rows * self.ff * w}

    def tolerance(self):
        # with its sums in another order, the router may take another of two experts that are all but equal for a token
        return {"rel": 1e-2, "max": 0.95}


KINDS = {"qwen3": Qwen3, "pooled": Pooled, "gla": Gla, "latent": Latent, "sink": Sink, "talk": Talk, "ssd": Ssd, "experts": Experts}


def built(module, *args, **kwargs):
    """A module with bf16 parameters on the GPU, as the model runner builds them."""
    default = torch.get_default_dtype()
    torch.set_default_dtype(BF16)
    try:
        with torch.device(DEV):
            return module(*args, **kwargs).to(DEV)
    finally:
        torch.set_default_dtype(default)


class State:
    """What a program has in hand before a step: layer, inputs, metadata; for a decode step the captured graph."""

    @torch.inference_mode()
    def __init__(self, case, seed):
        self.kind = KINDS[case["kind"]](case, seed)
        self.layer = self.kind.layer()
        self.kind.metadata()
        self.graph = None
        if case["step"] == "decode":
            held = [(t, t.clone()) for t in self.changed()]
            self.pass_()                               # allocates the kernels' workspaces
            self.graph = torch.cuda.CUDAGraph()
            with torch.cuda.graph(self.graph):
                self.outputs = self.pass_()
            for t, before in held:
                t.copy_(before)

    def changed(self):
        """What a pass updates from its own earlier value."""
        named = [getattr(self.layer, "state", None), getattr(self.layer, "ring", None), *(getattr(self.layer, "rings", None) or [])]
        return [t for t in named + [getattr(self.kind, "x", None)] if t is not None]

    @torch.inference_mode()
    def pass_(self):
        self.kind.publish()
        out = self.kind.call(self.layer)
        reset_context()
        return out


def prepare(case, seed):
    return State(case, seed)


def run(state):
    if state.graph is None:
        return state.pass_()
    state.graph.replay()
    return state.outputs


def work(case):
    return KINDS[case["kind"]](case).work()


def tolerance(case):
    return KINDS[case["kind"]](case).tolerance()


@torch.inference_mode()
def exact(case, seed):
    return KINDS[case["kind"]](case, seed).exact()
