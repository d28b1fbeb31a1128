"""Tibenex on the CPU: the plain implementation against closed forms, planted mistakes, configuration and checkpoint routing,
tables, the host side of caches and state slots, and argument checks of the entry points."""
import copy
import ctypes
import json
import math

import pytest
import torch

from oracle import tibenex as O
from tests import tibenex_cases as C
from tinyllmforge_amd.config import NO_WINDOW, Config, TibenexConfig, model_config
from tinyllmforge_amd.engine.scheduler import Scheduler
from tinyllmforge_amd.engine.sequence import Sequence
from tinyllmforge_amd.sampling_params import SamplingParams

F64 = torch.float64
t64 = lambda *v: torch.tensor(v, dtype=F64)


# ---------------------------------------------------------------------------------------------- plain implementation
def test_norms_closed_form():
    x = t64([3.0, 4.0, 1.0, 7.0])
    assert torch.allclose(O.rms_norm(x, t64(1.0, 2.0, 1.0, 0.5), 0.25), t64([3, 8, 1, 3.5]) / math.sqrt(75 / 4 + 0.25))
    a, b = math.sqrt(25 / 2 + 0.5), math.sqrt(50 / 2 + 0.5)
    assert torch.allclose(O.grouped_rms_norm(x, t64(1.0, 1.0, 2.0, 1.0), 2, 0.5), t64([3 / a, 4 / a, 2 / b, 7 / b]))
    y = O.post_norm(t64([1.0, 2.0]), t64([10.0, 20.0]), 3.0, t64(0.1, 0.5), t64(1.0, 2.0), 0.0)       # sums 4 and 16
    assert torch.allclose(y, t64([4.0, 32.0]) / math.sqrt(136))


def test_token_shift_reads_the_row_before_as_it_was():
    x = t64([1.0, 10.0], [2.0, 20.0], [4.0, 40.0])
    assert torch.allclose(O.token_shift(x, t64(0.25, 1.0)), t64([0.75, 0.0], [1.75, 10.0], [3.5, 20.0]))


def test_convolution_looks_back():
    u, w = t64([1.0], [10.0], [100.0], [1000.0]), t64([0.5, 2.0, 3.0])      # two back, one back, the token itself
    assert O.causal_conv(u, w, t64(0.25))[:, 0].tolist() == [3.25, 32.25, 320.75, 3205.25]


def test_rotations_closed_form():
    rot, x = dict(dims=4, base=100.0), torch.arange(1.0, 7.0, dtype=F64).view(1, 1, 6)
    c, s, c1, s1 = math.cos(3), math.sin(3), math.cos(.3), math.sin(.3)
    assert O.rotate_halves(x, [3], rot)[0, 0].tolist() == pytest.approx([c - 3 * s, 2 * c1 - 4 * s1, 3 * c + s, 4 * c1 + 2 * s1, 5, 6])
    assert O.rotate_neighbours(x, [3], rot)[0, 0].tolist() == pytest.approx([c - 2 * s, 2 * c + s, 3 * c1 - 4 * s1, 4 * c1 + 3 * s1, 5, 6])


def test_scaled_frequencies():
    rot = dict(dims=16, base=1000.0, scaling=dict(factor=4.0, original=100, fast=10.0, slow=1.0))
    pair = lambda t: 16 * math.log(100 / (2 * math.pi * t)) / (2 * math.log(1000))
    assert (math.floor(pair(10)), math.ceil(pair(1))) == (0, 4)
    f, mult = O.rotation_frequencies(rot)
    ramp = [0, .25, .5, .75, 1, 1, 1, 1]
    assert f == pytest.approx([1000 ** (-i / 8) * ((1 - r) + r / 4) for i, r in enumerate(ramp)]) and mult == pytest.approx(0.1 * math.log(4) + 1)


def test_talking_attention_closed_form():
    T = 3
    q, k, v = torch.zeros(T, 2, 2, dtype=F64), torch.zeros(T, 1, 2, dtype=F64), t64(1.0, 4.0, 10.0).view(T, 1, 1)
    k[0, 0, 0], q[2, 1, 0] = 2.0, 3.0
    o = O.talking_attention(q, k, v, 0.5, t64(1.0, 0.4), t64([1.0, 0.0], [0.5, -2.0]))
    e = math.exp(1.2)
    own = [[1, 2.5, 5], [1, 2.5, (e + 14) / (e + 2)]]                            # what the heads see on their own
    assert o[:, 0, 0].tolist() == pytest.approx(own[0])
    assert o[:, 1, 0].tolist() == pytest.approx([0.5 * a - 2 * b for a, b in zip(*own)])


def test_state_space_closed_form():
    x, B, Cc = t64([2.0], [3.0]).view(2, 1, 1), t64([1.0, 4.0], [0.0, 1.0]).view(2, 1, 2), t64([1.0, 1.0], [1.0, 2.0]).view(2, 1, 2)
    y = O.state_space_scan(x, B, Cc, t64([0.5], [2.0]), t64(math.log(0.3)), t64(7.0))
    s = [1.0, 4.0]                                               # 0.5 * B * 2
    s2 = [s[0] * math.exp(-0.6), s[1] * math.exp(-0.6) + 6]
    assert y.flatten().tolist() == pytest.approx([5 + 14, s2[0] + 2 * s2[1] + 21])
    assert O.softplus(t64(0.0, 50.0, -2.0)).tolist() == pytest.approx([math.log(2), 50, math.log1p(math.exp(-2))])


def test_a_head_reads_its_group():
    """Four heads on two groups: heads 0, 1 read the first one."""
    g = torch.Generator().manual_seed(0)
    r = lambda *s: torch.randn(*s, generator=g, dtype=F64)
    x, B, Cc, dt = r(5, 4, 3), r(5, 2, 6), r(5, 2, 6), r(5, 4).abs()
    A, D = r(4), r(4)
    y = O.state_space_scan(x, B, Cc, dt, A, D)
    for h, grp in ((0, 0), (1, 0), (2, 1), (3, 1)):
        one = O.state_space_scan(x[:, h:h + 1], B[:, grp:grp + 1], Cc[:, grp:grp + 1], dt[:, h:h + 1], A[h:h + 1], D[h:h + 1])
        assert torch.allclose(y[:, h], one[:, 0])


def plant(monkeypatch, cfg, w, fault):
    """``(configuration, weights)`` with a mistake, or the mistake put into the plain implementation."""
    cfg, w = copy.deepcopy(cfg), dict(w)
    change = lambda end, f: w.update({n: f(x) for n, x in w.items() if n.endswith(end)})
    put = lambda name, f: monkeypatch.setattr(O, name, f(getattr(O, name)))
    mixers = [la["mixer"] for la in cfg["layers"]]
    cut = lambda real: lambda u, *a: torch.cat([real(u[:64], *a), real(u[64:], *a)])
    if fault == "no shift":
        change("shift", lambda x: 0 * x)
    elif fault == "shift forgets at 64":
        put("token_shift", cut)
    elif fault == "shift reads shifted rows":
        def chained(x, mix):
            out, before = [], torch.zeros_like(x[0])
            for row in x:
                before = row + (before - row) * mix
                out.append(before)
            return torch.stack(out)
        monkeypatch.setattr(O, "token_shift", chained)
    elif fault == "first row shifted towards itself":
        monkeypatch.setattr(O, "token_shift", lambda x, mix: x + (torch.cat([x[:1], x[:-1]]) - x) * mix)
    elif fault == "no layer scale":
        change("ls1", lambda x: 0 * x + 1)
    elif fault == "no layer scale behind the feed-forward":
        change("ls2", lambda x: 0 * x + 1)
    elif fault == "alpha left out":
        cfg["postln_alpha"] = 1.0
    elif fault == "layer scale on the stream":
        put("post_norm", lambda real: lambda x, y, a, ls, wt, eps: real(x, y + a * x, 0.0, ls, wt, eps))
    elif fault == "embedding not scaled":
        cfg["embedding"]["scale"] = 1.0
    elif fault == "taps reversed":
        change("conv", lambda x: x.flip(-1))
    elif fault == "convolution forgets at 64":
        put("causal_conv", cut)
    elif fault == "no convolution bias":
        change("conv.b", lambda x: 0 * x)
    elif fault == "state forgets at 64":
        put("state_space_scan", lambda real: lambda x, B, Cc, dt, A, D: torch.cat(
            [real(x[:64], B[:64], Cc[:64], dt[:64], A, D), real(x[64:], B[64:], Cc[64:], dt[64:], A, D)]))
    elif fault == "no D":
        change(".D", lambda x: 0 * x)
    elif fault == "step not softplus":
        monkeypatch.setattr(O, "softplus", lambda z: z.clamp(min=0))
    elif fault == "no step bias":
        change("dt_bias", lambda x: 0 * x)
    elif fault == "groups taken in turn":
        def turn(x, B, Cc, dt, A, D):
            G = B.shape[1]
            order = [h for g in range(G) for h in range(g, x.shape[1], G)]
            y = torch.zeros_like(x)
            y[:, order] = real(x[:, order], B, Cc, dt[:, order], A[order], D[order])
            return y
        real = O.state_space_scan
        monkeypatch.setattr(O, "state_space_scan", turn)
    elif fault == "norm over all groups at once":
        put("grouped_rms_norm", lambda real: lambda x, wt, groups, eps: real(x, wt, 1, eps))
    elif fault == "heads do not mix":
        change("talk", lambda x: torch.eye(x.shape[0], dtype=x.dtype))
    elif fault == "mix transposed":
        change("talk", lambda x: x.T.contiguous())
    elif fault == "mixed before the softmax":
        def early(q, k, v, scale, temp, talk):
            H, share = q.shape[1], q.shape[1] // k.shape[1]
            s = torch.stack([q[:, h] @ k[:, h // share].T * scale * temp[h] for h in range(H)])
            wt = O.causal_weights(torch.tensordot(talk, s, 1))
            return torch.stack([wt[h] @ v[:, h // share] for h in range(H)], dim=1)
        monkeypatch.setattr(O, "talking_attention", early)
    elif fault == "no temperature":
        change("temp", lambda x: 0 * x + 1)
    elif fault == "query norm head by head":
        def by_heads(x, wt, eps):
            heads = {m["heads"] * m["dim"]: m["heads"] for m in mixers if "kv_heads" in m}
            return real(x, wt, eps) if x.shape[-1] not in heads else O.grouped_rms_norm(x, wt, heads[x.shape[-1]], eps)
        real = O.rms_norm
        monkeypatch.setattr(O, "rms_norm", by_heads)
    elif fault == "one plus the weight":
        change("k.norm", lambda x: 1 + x)
    elif fault == "halves for neighbours":
        monkeypatch.setattr(O, "rotate_neighbours", O.rotate_halves)
    elif fault == "neighbours for halves":
        monkeypatch.setattr(O, "rotate_halves", O.rotate_neighbours)
    elif fault == "no scaling of the rotation":
        for m in mixers:
            m.get("rot", {}).pop("scaling", None)
    elif fault == "no factor on cos and sin":
        put("rotation_frequencies", lambda real: lambda rot: (real(rot)[0], 1.0))
    elif fault == "query latent not normed":
        ranks = {m["q_rank"] for m in mixers if "q_rank" in m}
        put("rms_norm", lambda real: lambda x, wt, eps: x * wt if wt.shape[0] in ranks else real(x, wt, eps))
    elif fault == "no head gate":
        change(".g", lambda x: 0 * x)
    elif fault == "keys from 48 back are lost":
        put("causal_weights", lambda real: lambda s: real(s.masked_fill(torch.ones_like(s, dtype=torch.bool).tril(-48), -1e9)))
    elif fault == "a token does not see itself":
        own = lambda s: s.masked_fill(torch.eye(s.shape[-1], dtype=torch.bool) & (torch.arange(s.shape[-1]) > 0), -1e9)
        put("causal_weights", lambda real: lambda s: real(own(s)))
    else:
        raise KeyError(fault)
    return cfg, w


FAULTS = ["no shift", "shift forgets at 64", "shift reads shifted rows", "first row shifted towards itself", "no layer scale",
          "no layer scale behind the feed-forward", "alpha left out", "layer scale on the stream", "embedding not scaled", "taps reversed",
          "convolution forgets at 64", "no convolution bias", "state forgets at 64", "no D", "step not softplus", "no step bias",
          "groups taken in turn", "norm over all groups at once", "heads do not mix", "mix transposed", "mixed before the softmax",
          "no temperature", "query norm head by head", "one plus the weight", "halves for neighbours", "neighbours for halves",
          "no scaling of the rotation", "no factor on cos and sin", "query latent not normed", "no head gate", "keys from 48 back are lost",
          "a token does not see itself"]


@pytest.mark.parametrize("fault", FAULTS)
def test_the_tests_weights_show_a_fault(fault, monkeypatch):
    """A mistake planted in the plain implementation is far above the GPU tests' tolerances."""
    cfg = C.CONFIGS["odd"]
    w, toks = C.weights(cfg), C.tokens(cfg, 80)
    want = O.forward(cfg, w, toks)
    err = C.logit_error(O.forward(*plant(monkeypatch, cfg, w, fault), toks), want)
    assert err.max() > 0.02          # 32-bit runs are held to 5e-5


# ---------------------------------------------------------------------------------------------- configuration, loading
def test_registry_and_config(tmp_path):
    from tinyllmforge_amd.models.registry import model_class
    from tinyllmforge_amd.models.tibenex import TibenexForCausalLM
    cfg = C.CONFIGS["odd"]
    (tmp_path / "config.json").write_text(json.dumps(cfg))
    hf = model_config(str(tmp_path))
    assert isinstance(hf, TibenexConfig) and model_class(hf) is TibenexForCausalLM
    assert hf.postln_alpha == 1.6 and hf.embedding_scale == 5.0 and hf.hidden_size == 90 and hf.vocab_size == 203 and hf.norm["eps"] == 1e-3
    assert hf.portioned and hf.recurrent and hf.float32 and hf.windows == (NO_WINDOW,)
    assert not model_config(C.config(64, 64, [C.attention(1, 1, 8, 8, 4)])).windows            # no latent cache, no window
    c = Config(str(tmp_path), max_model_len=300, kvcache_block_size=64, max_num_batched_tokens=64, dtype="float32")
    assert c.hf_config.torch_dtype == torch.float32 and c.hf_config.max_position_embeddings == 300
    for where, value in ((("layers", 0, "type"), "other"), (("layers", 0, "mixer", "groups"), 4), (("layers", 0, "mixer", "norm_groups"), 7),
                         (("layers", 1, "mixer", "kv_heads"), 4), (("layers", 1, "mixer", "rot", "dims"), 22), (("layers", 2, "mixer", "rot", "dims"), 4),
                         (("layers", 1, "mlp", "kind"), "moe"), (("layers", 0, "mixer", "conv"), 0)):
        bad = copy.deepcopy(cfg)
        at = bad
        for k in where[:-1]:
            at = at[k]
        at[where[-1]] = value
        with pytest.raises(AssertionError):
            model_config(bad)


def build(cfg, dtype=torch.bfloat16, positions=32):
    from tinyllmforge_amd.models.tibenex import TibenexForCausalLM
    hf = model_config(copy.deepcopy(cfg))
    hf.max_position_embeddings, hf.torch_dtype = positions, dtype
    torch.set_default_dtype(dtype)
    try:
        return TibenexForCausalLM(hf)
    finally:
        torch.set_default_dtype(torch.float32)


def test_loading_fills_every_parameter(tmp_path):
    from safetensors.torch import save_file
    from tinyllmforge_amd.utils.loader import load_model, load_state_dict
    for name, cfg in C.CONFIGS.items():
        assert build(cfg).expected_tensors() == set(C.shapes(cfg)), name
    cfg = C.CONFIGS["odd"]
    w, model = C.weights(cfg), build(cfg)
    save_file(w, str(tmp_path / "model.safetensors"))
    load_model(model, str(tmp_path))
    la = model.layers[0]
    assert torch.equal(la.shift.weight, w["l0.shift"]) and la.shift.embed_scale == 5.0 and la.norm1.alpha == 1.6
    assert torch.equal(la.norm1.layer_scale, w["l0.ls1"]) and torch.equal(la.norm2.layer_scale, w["l0.ls2"]) and torch.equal(la.norm2.weight, w["l0.norm2"])
    s = la.mix.ssd
    assert torch.equal(s.conv, w["l0.mix.conv"].T) and torch.equal(s.conv_bias, w["l0.mix.conv.b"]) and torch.equal(s.A_log, w["l0.mix.A_log"])
    assert torch.equal(s.dt_bias, w["l0.mix.dt_bias"]) and torch.equal(s.D, w["l0.mix.D"]) and torch.equal(s.norm.weight, w["l0.mix.norm"])
    assert torch.equal(la.mix.inp.weight[:s.columns, :90], w["l0.mix.in"]) and s.norm_groups == 4
    at, mix = 0, model.layers[1].mix
    for part, rows in (("q", 120), ("k", 60), ("v", 39)):
        assert torch.equal(mix.qkv.weight[at:at + rows, :90], w["l1.mix." + part])
        at += rows
    assert torch.equal(mix.attn.talk, w["l1.mix.talk"]) and torch.equal(mix.attn.temp, w["l1.mix.temp"]) and torch.equal(mix.attn.k_norm.weight, w["l1.mix.k.norm"])
    mix = model.layers[2].mix
    for part in ("dq", "dkv", "g"):
        rows = w["l2.mix." + part].shape[0]
        assert torch.equal(mix.down.weight[mix.down.offset(part):mix.down.offset(part) + rows, :90], w["l2.mix." + part])
    assert torch.equal(mix.q_norm.weight, w["l2.mix.dq.norm"]) and torch.equal(mix.uq.weight[:51, :17], w["l2.mix.uq"])
    assert torch.equal(mix.attn.uk, w["l2.mix.uk"].view(mix.attn.uk.shape)) and mix.attn.halves
    assert model.layers[3].mlp is None and torch.equal(model.head.weight[:203, :90], w["head"])
    other = build(cfg)
    load_state_dict(other, w)
    assert all(torch.equal(a, b) for a, b in zip(model.layers.parameters(), other.layers.parameters()))
    with pytest.raises(ValueError, match="l2.mix.dq.norm"):
        load_state_dict(build(cfg), {k: v for k, v in w.items() if k != "l2.mix.dq.norm"})
    for tensor in ("l9.norm1", "l0.mlp.router", "l3.norm2", "l3.ls2", "l1.mix.g", "l0.mix.talk"):
        with pytest.raises(KeyError):
            model.route_tensor(tensor)


def test_random_initialisation_keeps_norms():
    from tinyllmforge_amd.utils.loader import random_init_
    model = random_init_(build(C.CONFIGS["odd"]), seed=3)
    assert (model.layers[0].norm1.weight == 1).all() and (model.norm.weight == 1).all() and (model.layers[1].mix.attn.q_norm.weight == 1).all()
    assert (model.layers[2].mix.q_norm.weight == 1).all() and model.layers[0].mix.ssd.conv.any()


def test_tables_agree_with_the_plain_implementation():
    from tinyllmforge_amd.layers.rotary_embedding import rotation_table
    for rot in (C.CONFIGS["odd"]["layers"][2]["mixer"]["rot"], C.CONFIGS["odd"]["layers"][1]["mixer"]["rot"],
                dict(dims=8, base=1e6, scaling=dict(factor=2.0, original=10, fast=500.0, slow=300.0))):
        t = rotation_table(rot["dims"], 9000, rot["base"], **(rot.get("scaling") or {}))
        f, mult = O.rotation_frequencies(rot)
        for p in (0, 1, 77, 8999):
            want = [math.cos(p * x) * mult for x in f] + [math.sin(p * x) * mult for x in f]
            assert t[p].tolist() == pytest.approx(want, abs=1e-6)
    model = build(C.CONFIGS["even"], positions=64)
    a, b, c = (model.layers[i].mix.attn.cos_sin for i in (0, 1, 3))
    assert a.shape == (64, 32) and b.shape == (64, 32) and a.data_ptr() == c.data_ptr() and a.data_ptr() != b.data_ptr()


def test_pages_and_states_of_a_layer():
    model = build(C.CONFIGS["odd"])
    item, (a, b, c) = 2, (model.layers[i] for i in range(3))
    inner, chan = 60, 60 + 2 * 3 * 13
    assert a.shift.slot_bytes() == 4 * 2 * 90 and a.mix.ssd.slot_bytes() == 4 * 6 * 13 * 10 + 3 * chan * item
    assert b.mix.attn.page_bytes(64) == 64 * 3 * (32 + 32) * item
    assert c.mix.attn.page_bytes(64) == 64 * 64 * item                           # 21 latent channels and 6 rotated ones, padded
    a.shift.bind_slots(3, "cpu")
    a.mix.ssd.bind_slots(3, "cpu")
    b.mix.attn.bind_pages(2, 64, "cpu")
    assert a.shift.ring.shape == (3, 2, 90) and a.shift.ring.dtype == a.mix.ssd.state.dtype == torch.float32
    assert a.mix.ssd.state.shape == (3, 6, 13, 10) and a.mix.ssd.ring.shape == (3, 3, chan) and b.mix.attn.kv.k.shape == (2, 3, 64, 32)
    a.shift.bind_slots(0, "cpu")
    a.mix.ssd.bind_slots(0, "cpu")
    b.mix.attn.bind_pages(0, 64, "cpu")
    assert a.shift.ring is None and a.mix.ssd.state is None and b.mix.attn.kv is None and a.mix.ssd.columns == inner + chan + 6


def test_scheduler_hands_out_state_slots():
    cfg = Config(C.CONFIGS["ones"], max_model_len=512, kvcache_block_size=64, max_num_batched_tokens=48, max_num_seqs=4,
                 num_kvcache_blocks=6, num_state_slots=2)
    Sequence.block_size = 64
    s = Scheduler(cfg)
    for n in (5, 9, 7):
        s.add(Sequence([1] * n, SamplingParams(0.0, 3, True)))
    slots = set()
    while not s.is_finished():
        batch, _ = s.schedule()
        assert len(batch) <= 2 and len({q.state_slot for q in batch}) == len(batch)
        slots |= {q.state_slot for q in batch}
        ends = [q.num_computed + q.num_scheduled == len(q) for q in batch]
        s.postprocess(batch, [7 if e else None for e in ends])
    assert slots == {0, 1} and len(s.state_slots.free) == 2 and len(s.block_manager.free_block_ids) == 6


# ---------------------------------------------------------------------------------------------- argument checks
def test_entry_points_reject_bad_arguments_on_the_host():
    from tinyllmforge_amd import _lib
    lib, a = _lib.load(), 4096
    NULL, SHAPE, WORK, TYPE = -1, -2, -4, -5
    post = lambda y=a, ys=64, splits=1, p=None, ls=a, x=a, out=8192, mix=None, ring=None, slots=4, st=None, rs=None, cu=None, pos=None, nxt=None, \
        h=None, rows=2, width=64, dt=0: lib.tlf_post_rmsnorm(y, ys, p, splits, None, ls, 1.0, x, a, 1e-6, out, mix, ring, slots, st, rs, cu, pos, nxt,
                                                             h, rows, width, dt, None)
    shift = dict(mix=a, ring=a, st=a, pos=a, h=a)
    assert post(ls=None) == NULL and post(ys=32) == SHAPE and post(rows=0) == 0 and post(width=20000, ys=20000) == SHAPE and post(dt=9) == TYPE
    assert post(**{**shift, "ring": None}) == NULL and post(**{**shift, "h": None}) == NULL and post(**shift, nxt=a) == TYPE
    assert post(**shift, rs=a, cu=a, out=a) == TYPE and post(**shift, rs=a) == NULL and post(nxt=a) == NULL      # portions not in place
    emb = lambda vocab=9, mix=a, width=64, rows=2, x=a, dt=0, ids=a: lib.tlf_embed_shift(ids, a, vocab, 1.0, x, mix, a, 4, a, None, None, a, a, rows, width, dt, None)
    assert emb(ids=None) == NULL and emb(vocab=0) == SHAPE and emb(width=0) == SHAPE and emb(rows=0) == 0 and emb(x=None) == NULL and emb(dt=5) == TYPE
    rows = lambda cols=60, groups=4, xs=60, os=64, w=a, dt=0, n=2: lib.tlf_rows_rmsnorm(a, xs, w, a, os, n, cols, groups, 1e-6, dt, None)
    assert rows(groups=7) == SHAPE and rows(xs=50) == SHAPE and rows(os=50) == SHAPE and rows(w=None) == NULL and rows(dt=4) == TYPE and rows(n=0) == 0

    shape = (6, 3, 20, 13)                 # heads, kv heads, dim, value dim: 120 + 60 + 39 columns
    prep = lambda sizes=shape, ld=224, q=a, n=2, sp=1, p=None, rot=12, cos=a, bs=64, dt=0: lib.tlf_talk_prep(
        a, ld, p, sp, None, a, a, a, a, cos, 10, rot, a, q, a, a, n, *sizes, bs, 5, 1e-6, 0.1, dt, None)
    assert prep(q=None) == NULL and prep(ld=210) == SHAPE and prep(n=0) == 0 and prep(rot=22) == SHAPE and prep(rot=3) == SHAPE and prep(cos=None) == NULL
    assert prep(bs=100) == SHAPE and prep(sizes=(6, 4, 20, 13)) == SHAPE and prep(sizes=(1100, 1, 32, 13), ld=99999) == SHAPE and prep(dt=7) == TYPE
    assert prep(sp=3) == NULL
    att = lambda sizes=shape, ldo=78, bt=4, most=200, out=a, ws=None, nb=0, dt=0, n=2, talk=a: lib.tlf_talk_attn_rows(
        a, a, a, a, bt, a, a, None, talk, out, ldo, n, *sizes, 64, most, 10, dt, ws, nb, None)
    assert att(ldo=70) == SHAPE and att(bt=3) == SHAPE and att(out=None) == NULL and att(talk=None) == NULL and att() == WORK and att(dt=3) == TYPE
    assert att(n=0) == 0 and att(n=70000) == SHAPE and att(sizes=(1025, 1, 20, 13), ldo=99999) == SHAPE
    size = lambda *v: lib.tlf_talk_attn_rows_workspace_bytes(*v)
    assert size(0, *shape, 200, 0) == 0 and size(2, *shape, 200, 0) >= 2 * 6 * 200 * 4 and att(ws=a, nb=size(2, *shape, 200, 0) - 1) == WORK
    pre = lambda sizes=shape, ldo=78, out=a, n=1, stats=a: lib.tlf_talk_attn_prefill(a, a, a, a, 4, a, a, 0, n, 8, a, stats, out, ldo, *sizes, 64, 10, None)
    assert pre(ldo=70) == SHAPE and pre(out=None) == NULL and pre(stats=None) == NULL and pre(n=0) == 0 and pre(sizes=(3, 1, 140, 13)) == TYPE
    room = lambda n=1, most=8, keys=256, sizes=shape: lib.tlf_talk_attn_prefill_workspace_bytes(n, most, keys, *sizes)
    assert room() > 0 and room(keys=96) == 0 and room(n=0) == 0 and room(n=600) == 0 and room(sizes=(33, 1, 20, 13)) == 0
    cut = lambda ws=None, nb=0, ldo=78, out=a, n=1: lib.tlf_talk_attn_prefill_cut(a, a, a, a, 4, a, a, 0, n, 8, a, a, out, ldo, *shape, 64, 10, ws, nb, None)
    assert cut() == WORK and cut(ws=a, nb=room() - 1) == WORK and cut(ldo=70) == SHAPE and cut(out=None) == NULL and cut(n=0) == 0
    pays = lambda n=1, most=5000, rows=5000, keys=5056, sizes=(16, 8, 128, 128): lib.tlf_talk_attn_prefill_cuts(n, most, rows, 0, keys, *sizes)
    assert pays() == 1 and pays(n=0) == 0 and pays(most=0) == 0 and pays(sizes=(33, 1, 64, 64)) == 0 and pays(n=24, most=250, rows=6000, keys=256) == 0
    load = (ctypes.c_int64 * 10)(64, 4, 256, 256 * 1026, 1028)       # the second half: no long ones
    route = lambda s=load, sizes=(16, 8, 128, 128): lib.tlf_talk_attn_prefill_route(0, s, ctypes.byref(load, 40), *sizes)
    assert route() == 1 and route(s=None) == 0 and route(sizes=(33, 1, 64, 64)) == 0
    assert lib.tlf_talk_attn_prefill_tile_rows(16, 8, 128, 128) == 32 and lib.tlf_talk_attn_prefill_tile_rows(33, 1, 64, 64) == 0
    ok = lib.tlf_talk_attn_prefill_supported
    assert ok(32, 8, 128, 128) == 1 and ok(33, 1, 64, 64) == 0 and ok(4, 2, 129, 64) == 0 and ok(4, 2, 64, 129) == 0 and ok(1, 1, 1, 1) == 1

    ssd = (4, 12, 20, 2)                   # heads, value dim, state, groups: 48 + 48 + 80 + 4 columns
    dec = lambda sizes=ssd, ld=180, ring=a, out=a, ldo=48, taps=3, n=2, dt=0, sp=1, p=None, slots=4: lib.tlf_ssd_decode(
        a, ld, p, sp, None, a, a, taps, a, a, a, ring, a, a, slots, a, out, ldo, n, *sizes, dt, None)
    assert dec(ring=None) == NULL and dec(ld=170) == SHAPE and dec(ldo=40) == SHAPE and dec(taps=0) == SHAPE and dec(n=0) == 0 and dec(dt=8) == TYPE
    assert dec(sizes=(4, 12, 20, 3)) == SHAPE and dec(sizes=(4, 12, 600, 2), ld=9999) == SHAPE and dec(sp=2) == NULL
    por = lambda sizes=ssd, ld=180, out=a, ldo=48, ws=None, nb=0, n=5, most=5, dt=0: lib.tlf_ssd_portions(
        a, ld, a, a, 3, a, a, a, a, a, a, 4, a, a, a, a, 0, 1, 0, most, out, ldo, n, *sizes, dt, ws, nb, None)
    need = lib.tlf_ssd_portions_workspace_bytes(5, 1, 5, *ssd, 0)
    assert need > 0 and por(out=None) == NULL and por(ld=170) == SHAPE and por() == WORK and por(ws=a, nb=need - 1) == WORK and por(dt=8) == TYPE
    assert por(n=0) == 0 and por(sizes=(4, 12, 20, 3)) == SHAPE
    lat = lambda halves=1, q=None, cache=a, cq=a, cqn=a, stride=64, gate=a, ld=80, dt=0, sizes=(3, 11, 6, 21, 9): lib.tlf_latent_prep(
        a, ld, None, 1, None, 17, a, a, a, 10, halves, a, 99, q, cache, 0, 17, cqn, cq, stride, 44, gate, 2, *sizes, 1e-6, dt, None)
    assert lat(cache=None) == NULL and lat(cq=None) == NULL and lat(stride=16) == SHAPE and lat(ld=40) == SHAPE and lat(dt=9) == TYPE


@pytest.mark.parametrize("sizes,seqs,tokens,segments", [((32, 64, 128, 1), 1, 2000, 8), ((32, 64, 128, 1), 1, 4000, 16), ((32, 64, 128, 1), 6, 520, 1),
                                                        ((16, 64, 128, 1), 1, 4000, 15), ((32, 64, 64, 1), 1, 1500, 12), ((128, 64, 128, 8), 4, 3000, 4)])
def test_few_state_space_groups_keep_a_head_per_workgroup(sizes, seqs, tokens, segments):
    """Their segments are of at least four chunks, so there are fewer of them than the heads of a group together would need; what a segment
    leaves behind is in the workspace."""
    from tinyllmforge_amd import _lib
    (H, P, N, G), rows, up = sizes, seqs * tokens, lambda v: -(-v // 256) * 256
    parts = seqs * segments * H if segments > 1 else 0
    want = up(2 * rows * (H * P + 2 * G * N)) + 2 * up(4 * rows * H) + up(4 * parts) + up(4 * parts * N * P)
    assert _lib.load().tlf_ssd_portions_workspace_bytes(rows, seqs, tokens, *sizes, 0) == want
