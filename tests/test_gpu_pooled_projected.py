"""Portions of pooled-window attention whose queries are made where they are read, against the separate preparation."""
from types import SimpleNamespace

import numpy as np
import pytest
import torch

from tinyllmforge_amd import ops
from tinyllmforge_amd.engine.inputs import portion_inputs
from tinyllmforge_amd.layers.pooled_attention import PooledWindowAttention
from tinyllmforge_amd.layers.rotary_embedding import rotation_table
from tinyllmforge_amd.utils.context import reset_context, set_portions_context

BF16 = torch.bfloat16


class Sized(SimpleNamespace):
    def __len__(self):
        return self.size


def layer_of(H, G, D, rot, size, pool, pages, seed, scale):
    g = torch.Generator().manual_seed(seed)
    layer = PooledWindowAttention(H, G, D, scale, size, pool, rot, rotation_table(rot, 2048, 1e4).cuda(), 1e-6, BF16)
    layer.score_bias.data = torch.randn(H, generator=g).to(BF16).cuda() - 2
    layer.bind_pages(pages, 64, "cuda")
    for t in (layer.kv.k, layer.kv.v, layer.kv.pk, layer.kv.pv):
        t.fill_(3.0)
        t[..., D:] = 0
    return layer


def steps_of(lens, schedule):
    """Context fields of each step: ``schedule``: lists of (sequence, tokens), single tokens first."""
    rng = np.random.RandomState(len(lens))
    free = list(rng.permutation(sum(-(-n // 64) for n in lens) + 2))
    tables = [[int(free.pop()) for _ in range(-(-n // 64))] for n in lens]
    done = [0] * len(lens)
    for parts in schedule:
        seqs = [Sized(num_scheduled=n, num_computed=done[s], num_cached_tokens=done[s], num_cached_blocks=done[s] // 64, token_ids=range(done[s] + n),
                      last_token=0, block_table=tables[s][:-(-(done[s] + n) // 64)], state_slot=s, size=done[s] + n) for s, n in parts]
        fields = {k: torch.from_numpy(v).cuda() if isinstance(v, np.ndarray) else v for k, v in portion_inputs(seqs, 64, None, ()).items()}
        fields.pop("input_ids")
        for s, n in parts:
            done[s] += n
        yield fields


# heads, KV heads, dimensions, rotated ones, window, pool, biases
FORMS = [(4, 2, 40, 24, 37, 5, True), (8, 8, 128, 128, 64, 16, True), (6, 2, 64, 0, 100, 8, False), (20, 1, 96, 32, 130, 100, True),
         (2, 2, 8, 8, 1, 1, False), (32, 8, 128, 64, 80, 17, True), (9, 3, 32, 32, 20, 33, False)]


@pytest.mark.gpu
@pytest.mark.parametrize("H,G,D,rot,size,pool,biased", FORMS)
def test_projected_portions_are_the_prepared_ones(monkeypatch, H, G, D, rot, size, pool, biased):
    lens = [150, 67, 210]
    schedules = [[[(0, 150), (1, 67), (2, 210)]],
                 [[(0, 2), (1, 3)], [(0, 62), (2, 130)], [(0, 1), (1, 2), (2, 2)], [(0, 85), (1, 62), (2, 78)]],
                 [[(0, 100), (2, 64)], [(0, 1), (2, 1), (1, 20)], [(0, 1), (1, 1), (2, 145)], [(0, 48), (1, 46)]]]
    pages = sum(-(-n // 64) for n in lens) + 2
    width = -(-((H + G) * D + H) // 8) * 8 + 8                # rows of a wider array
    for i, schedule in enumerate(schedules):
        g = torch.Generator().manual_seed(i)
        r = lambda *s: torch.randn(*s, generator=g).to(BF16).cuda()
        qb, kb = (r(H * D), r(G * D)) if biased else (None, None)
        new, old = (layer_of(H, G, D, rot, size, pool, pages, i, 1.5 / D ** 0.5) for _ in range(2))
        for fields in steps_of(lens, schedule):
            positions = fields.pop("positions")
            proj = r(positions.numel(), width)[:, :(H + G) * D + H]
            outs, taken = [], []
            real = ops.pooled_attention_projected
            for layer, form in ((new, lambda *a: taken.append(real(*a)) or taken[-1]), (old, lambda *a: False)):
                monkeypatch.setattr(ops, "pooled_attention_projected", form)
                set_portions_context(**fields, max_len=256)
                outs.append(layer(proj, qb, kb, positions))
                reset_context()
            monkeypatch.undo()
            assert taken == [True]
            for name in ("k", "v", "pk", "pv"):
                assert torch.equal(getattr(new.kv, name), getattr(old.kv, name)), name
            assert torch.equal(outs[0], outs[1])


@pytest.mark.gpu
@pytest.mark.parametrize("pool", [3, 16, 17, 40])
def test_means_add_up_tokens_in_turn(pool):
    """Keys of two magnitudes that cancel: another order of a block's sum shows in its mean's first places."""
    H, G, D, lens = 4, 2, 64, [150, 67, 210]
    g = torch.Generator().manual_seed(pool)
    layers = [layer_of(H, G, D, 0, 40, pool, 12, 0, 0.1) for _ in range(2)]
    for fields in steps_of(lens, [[(0, 100), (1, 67), (2, 30)], [(0, 50), (2, 180)]]):
        positions = fields.pop("positions")
        proj = torch.randn(positions.numel(), (H + G) * D + 8, generator=g)
        keys = proj[:, H * D:(H + G) * D]
        keys[::3] *= 2.0 ** 20
        keys[1::3] = -keys[::3][:len(keys[1::3])]
        proj = proj.to(BF16).cuda()
        args = (fields["slot_mapping"], fields["block_tables"], fields["cu_seqlens_q"], fields["seq_starts"])
        slots, tables, cu, starts = args
        portions, most, rows = cu.numel() - 1, fields["max_portion"], proj[:, :(H + G) * D + H]
        for layer, projected in zip(layers, (True, False)):
            kv, out = layer.kv, torch.empty(len(proj), H * D, dtype=BF16, device="cuda")
            if projected:
                assert ops.pooled_attention_projected(rows, None, None, positions, layer.cos_sin, 0, slots, layer.score_bias.data, kv, tables, cu, starts, 0, portions,
                                                      most, 0.1, 1e-6, out)
            else:
                ops.attn_prep(rows, None, None, positions, layer.cos_sin, 0, slots, kv.k, kv.v, H, D, 1e-6)
                ops.pool_blocks(kv, tables, cu, starts, 0, portions, most)
    for name in ("k", "v", "pk", "pv"):
        assert torch.equal(getattr(layers[0].kv, name), getattr(layers[1].kv, name)), name


@pytest.mark.gpu
def test_weights_of_a_strongly_negative_bias():
    """2^-bias leaves the range of fp32 where 2^-(score + bias) does not: weights of 2^-90 and the like, not zeros."""
    H, G, D = 4, 2, 128
    fields = next(steps_of([150], [[(0, 150)]]))
    positions, g, outs = fields.pop("positions"), torch.Generator().manual_seed(5), []
    proj = torch.randn(150, (H + G) * D + 8, generator=g).to(BF16).cuda()
    proj[:, :G * D] = proj[:, H * D:(H + G) * D]               # heads 0 and 1 ask for their own token: scores of scale * D
    for projected in (True, False):
        layer = layer_of(H, G, D, 0, 40, 8, 8, 0, 0.25)
        layer.score_bias.data.copy_(torch.tensor([-89.0, -100.0, -60.0, 89.0]))
        out = torch.empty(150, H * D, dtype=BF16, device="cuda")
        args = (layer.kv, fields["block_tables"], fields["cu_seqlens_q"], fields["seq_starts"], 0, 1, 150)
        rows, slots, bias = proj[:, :(H + G) * D + H], fields["slot_mapping"], layer.score_bias.data
        if projected:
            assert ops.pooled_attention_projected(rows, None, None, positions, layer.cos_sin, 0, slots, bias, *args, 0.25, 1e-6, out)
        else:
            q, gate = ops.attn_prep(rows, None, None, positions, layer.cos_sin, 0, slots, layer.kv.k, layer.kv.v, H, D, 1e-6)
            ops.pool_blocks(*args)
            ops.pooled_attention_prefill(q, bias, gate, *args, 0.25, out)
        outs.append(out)
    assert torch.equal(*outs) and outs[0].view(150, H, D)[:, 0].any()


@pytest.mark.gpu
def test_rows_that_are_not_read_eight_at_a_time_are_prepared():
    """Refused, before anything is launched, and the layer prepares such rows apart."""
    fields = next(steps_of([70], [[(0, 70)]]))
    positions = fields.pop("positions")
    t = lambda *s: torch.randn(*s).to(BF16).cuda()
    for D, rot, width, first, bias, scale, takes in ((32, 32, 80, 0, 0, 0.2, True), (32, 32, 84, 0, 0, 0.2, False), (32, 32, 80, 4, 0, 0.2, False),
                                                     (32, 32, 80, 0, 4, 0.2, False), (32, 20, 80, 0, 0, 0.2, False), (36, 32, 120, 0, 0, 0.2, False),
                                                     (160, 32, 328, 0, 0, 0.2, False), (32, 32, 80, 0, 0, 2.1, True), (32, 32, 80, 0, 0, 2.2, True)):
        layer = layer_of(1, 1, D, rot, 20, 8, 5, 0, scale)
        proj, qb = t(71, width)[:, first:first + 2 * D + 1][:70], t(D + 8)[bias:bias + D]
        out = torch.full((70, D), 5.0, dtype=BF16, device="cuda")
        before = layer.kv.k.clone()
        args = (positions, layer.cos_sin, rot, fields["slot_mapping"], layer.score_bias.data, layer.kv, fields["block_tables"], fields["cu_seqlens_q"],
                fields["seq_starts"], 0, 1, 70, scale, 1e-6, out)
        assert ops.pooled_attention_projected(proj, qb, None, *args) == takes
        assert takes or ((out == 5).all() and torch.equal(layer.kv.k, before))
        set_portions_context(**fields, max_len=128)
        assert layer(proj, qb, None, positions).isfinite().all()
        reset_context()
