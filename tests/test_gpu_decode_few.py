"""Decode attention of a few sequences: shares of all lengths against fp64, and the projection's rows against its separate kernels."""
import pytest
import torch

from tinyllmforge_amd import ops

pytestmark = pytest.mark.gpu
BF, DEV = torch.bfloat16, "cuda"
EPS, SCALE = 1e-6, 128 ** -0.5


def step(ctxs, hq, hkv, bs, fp8, seed=0):
    """Caches that hold all but the newest tokens, tables with scattered pages, the newest tokens' projection."""
    g = torch.Generator().manual_seed(seed)
    need = [max(1, -(-c // bs)) for c in ctxs]
    pages = torch.randperm(sum(need) + 3, generator=g).tolist()
    bt = torch.full((len(ctxs), max(need) + 1), -1, dtype=torch.int32)
    for b, n in enumerate(need):
        bt[b, :n] = torch.tensor([pages.pop() for _ in range(n)])
    cache = lambda: torch.randn(sum(need) + 3, bs, hkv, 128, generator=g).to(BF)
    k, v = cache(), cache()
    scales = (None, None)
    if fp8:
        scales = torch.rand(hkv, generator=g) * 0.02 + 0.01, torch.rand(hkv, generator=g) * 0.02 + 0.01
        k, v = ((t.float() / s[:, None]).clamp(-448, 448).to(torch.float8_e4m3fn) for t, s in zip((k, v), scales))
        scales = tuple(s.to(DEV) for s in scales)
    slots = torch.tensor([bt[b, (c - 1) // bs] * bs + (c - 1) % bs if c else -1 for b, c in enumerate(ctxs)], dtype=torch.int32)
    qkv = torch.randn(len(ctxs), (hq + 2 * hkv) * 128, generator=g).to(BF)
    w = [(1 + 0.1 * torch.randn(128, generator=g)).to(BF).to(DEV) for _ in range(2)]
    angles = torch.rand(9000, 64, generator=g) * 6.3
    table = torch.cat([angles.cos(), angles.sin()], 1).to(DEV)
    return (qkv.to(DEV), k.to(DEV), v.to(DEV), torch.tensor(ctxs, dtype=torch.int32, device=DEV), bt.to(DEV), scales, slots.to(DEV), w, table,
            torch.tensor(ctxs, device=DEV))


def exact(q, k, v, ctxs, bt, hq, hkv, scales):
    q, k, v = q.double().view(len(ctxs), hq, 128), k.double(), v.double()
    if scales[0] is not None:
        k, v = k * scales[0].double()[:, None], v * scales[1].double()[:, None]
    out = torch.zeros_like(q)
    for b, c in enumerate(ctxs):
        if c == 0:
            continue
        at = torch.arange(c, device=DEV)
        page = bt[b].long()[at // k.shape[1]]
        rows = [torch.where((page >= 0)[:, None, None], t[page.clamp(min=0), at % k.shape[1]], 0.0).repeat_interleave(hq // hkv, 1) for t in (k, v)]
        w = torch.softmax(torch.einsum("hd,jhd->hj", q[b], rows[0]) * SCALE, -1)
        out[b] = torch.einsum("hj,jhd->hd", w, rows[1])
    return out.flatten(1)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,bs,ctxs", [
    (32, 8, 256, [700]), (32, 8, 16, [1, 64, 65, 0]), (32, 8, 256, [8000]), (16, 8, 256, [15, 16, 17, 63, 129, 1024, 1025, 2047]),
    (8, 8, 64, [4096, 1, 1000]), (64, 8, 256, [64, 3000]), (16, 2, 48, [1, 2, 500, 66]), (2, 2, 32, [4097]), (16, 16, 256, [300, 4095, 64, 65])])
def test_projection_rows_against_separate_kernels_and_fp64(hq, hkv, bs, ctxs, fp8):
    n = len(ctxs)
    assert ops.decode_few_supported(n, hq, hkv, 128, bs)
    qkv, k, v, ctx, bt, scales, slots, w, table, positions = step(ctxs, hq, hkv, bs, fp8)
    k2, v2 = k.clone(), v.clone()
    got = ops.decode_few(qkv, hq, k, v, ctx, bt, SCALE, *scales, (*w, EPS, positions, table, slots))
    q, _, _ = ops.qknorm_rope_store(qkv, *w, EPS, positions, table, hq, hkv, 128, k2, v2, slots, *scales)
    bits = lambda t: t.view(torch.uint8)
    assert torch.equal(bits(k), bits(k2)) and torch.equal(bits(v), bits(v2))
    assert torch.equal(got, ops.decode_few(q, hq, k2, v2, ctx, bt, SCALE, *scales))
    want = exact(q, k2, v2, ctxs, bt, hq, hkv, scales)
    # fp32 scores of up to 2^3 (off by 2^-20), weights and sums: the result is off by 2^-17 of the values' size; then half a bf16 ulp
    torch.testing.assert_close(got.double(), want, rtol=2 ** -8, atol=2 ** -13)


@pytest.mark.parametrize("hq,hkv,ctxs", [(32, 8, [700]), (32, 8, [8000, 1000, 2000, 5000]), (16, 8, [3000, 700, 64, 1500, 900, 2048, 333, 2999]), (64, 8, [4096]), (16, 16, [3000, 400])])
def test_results_are_no_further_from_64_bits_than_the_other_kernels(hq, hkv, ctxs):
    """The share of results that are not the nearest bfloat16 value: a layer's outputs may change by roundings where it takes the other kernel, and not more."""
    qkv, k, v, ctx, bt, _, _, _, _, _ = step(ctxs, hq, hkv, 256, False, seed=1)
    q = qkv[:, :hq * 128].contiguous()
    nearest = exact(q, k, v, ctxs, bt, hq, hkv, (None, None)).to(BF)
    off = lambda t: (t != nearest).double().mean().item()
    few, other = ops.decode_few(q, hq, k, v, ctx, bt, SCALE), ops.paged_decode_attention(q.view(len(ctxs), hq, 128), k, v, ctx, bt, SCALE)
    # fp32 weights against pairs of 16 bits: a result within 2^-17 of its values' size of a border may go either way, 2^-8 of them in bfloat16
    assert off(few) <= max(off(other), 2 ** -9) and off(few) < 2 ** -9


def test_rows_that_are_not_the_newest_token_come_from_the_cache():
    """Without a slot position context_len - 1 is read from the cache, with an earlier row's slot that row is the new one; an
    unmapped page reads as zeros; positions without cosines leave a head as normed."""
    ctxs, hq, hkv, bs = [70, 300, 128, 65], 8, 4, 64
    qkv, k, v, ctx, bt, scales, slots, w, table, positions = step(ctxs, hq, hkv, bs, False)
    slots[0], slots[1] = -1, k.shape[0] * bs
    slots[2] = bt[2, 0] * bs + 5
    bt[3, 0] = -1
    positions[3] = 9000
    k2, v2 = k.clone(), v.clone()
    got = ops.decode_few(qkv, hq, k, v, ctx, bt, SCALE, None, None, (*w, EPS, positions, table, slots))
    q, _, _ = ops.qknorm_rope_store(qkv, *w, EPS, positions, table, hq, hkv, 128, k2, v2, slots)
    assert torch.equal(k, k2) and torch.equal(v, v2)
    assert torch.equal(got, ops.decode_few(q, hq, k2, v2, ctx, bt, SCALE))
    torch.testing.assert_close(got.double(), exact(q, k2, v2, ctxs, bt, hq, hkv, (None, None)), rtol=2 ** -8, atol=2 ** -13)


def test_arrays_longer_than_the_rows_and_a_step_without_slots():
    """Static arrays of a larger batch, and rows that nothing keeps, as the separate kernels take them."""
    qkv, k, v, ctx, bt, _, slots, w, table, positions = step([70, 300, 5, 9], 16, 8, 64, False)
    few = lambda n, to: ops.decode_few(qkv[:2], 16, k, v, ctx[:n], bt[:n], SCALE, None, None, (*w, EPS, positions[:n], table, to))
    want = few(2, slots[:2])
    assert torch.equal(few(4, slots), want)
    k2, v2 = k.clone().normal_(), v.clone().normal_()
    k.copy_(k2), v.copy_(v2)
    got = few(2, None)
    q, _, _ = ops.qknorm_rope_store(qkv[:2], *w, EPS, positions[:2], table, 16, 8, 128, k2, v2, None)
    assert torch.equal(k, k2) and torch.equal(v, v2)
    assert torch.equal(got, ops.decode_few(q, 16, k2, v2, ctx[:2], bt[:2], SCALE)) and not torch.equal(got, want)


@pytest.mark.parametrize("fp8", [False, True])
@pytest.mark.parametrize("hq,hkv,bs,held", [(32, 8, 16, 14), (32, 8, 256, 700), (16, 8, 64, 62), (8, 8, 16, 127), (64, 8, 256, 5000), (2, 2, 32, 8000)])
def test_rows_of_one_sequence(hq, hkv, bs, held, fp8):
    """Three tokens of one sequence between two others: a row's attention sees the rows that the same call writes, behind edges of pages and shares."""
    n = 5 if hq // hkv <= 2 else 4
    longest, ctxs = held + 3, [held + 2, 70, held + 1, held + 3, 300][:n]
    mine = [0, 2, 3]
    qkv, k, v, ctx, bt, scales, slots, w, table, _ = step([longest if i in mine else c for i, c in enumerate(ctxs)], hq, hkv, bs, fp8, seed=held)
    bt[mine] = bt[0].clone()
    ctx, positions = torch.tensor(ctxs, dtype=torch.int32, device=DEV), torch.tensor(ctxs, device=DEV) - 1
    slots = (bt[torch.arange(n, device=DEV), positions // bs] * bs + positions % bs).to(torch.int32)
    k2, v2 = k.clone(), v.clone()
    got = ops.decode_few(qkv, hq, k, v, ctx, bt, SCALE, *scales, (*w, EPS, positions, table, slots))
    q, _, _ = ops.qknorm_rope_store(qkv, *w, EPS, positions, table, hq, hkv, 128, k2, v2, slots, *scales)
    bits = lambda t: t.view(torch.uint8)
    assert torch.equal(bits(k), bits(k2)) and torch.equal(bits(v), bits(v2))
    assert torch.equal(got, ops.decode_few(q, hq, k2, v2, ctx, bt, SCALE, *scales))
    torch.testing.assert_close(got.double(), exact(q, k2, v2, ctxs, bt, hq, hkv, scales), rtol=2 ** -8, atol=2 ** -13)


def test_replayed_with_other_lengths():
    """A captured step follows the lengths and tables it finds."""
    qkv, k, v, ctx, bt, _, slots, w, table, positions = step([4000, 90], 32, 8, 256, False)
    args = lambda: (qkv, 32, k, v, ctx, bt, SCALE, None, None, (*w, EPS, positions, table, slots))
    ops.decode_few(*args())
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = ops.decode_few(*args())
    for lens in ([4000, 90], [65, 0], [1, 4000], [64, 700]):
        ctx.copy_(torch.tensor(lens))
        slots.copy_(torch.tensor([bt[b, (c - 1) // 256] * 256 + (c - 1) % 256 if c and bt[b, (c - 1) // 256] >= 0 else -1 for b, c in enumerate(lens)]))
        graph.replay()
        replayed = out.clone()
        assert torch.equal(replayed, ops.decode_few(*args())), lens


@pytest.mark.parametrize("int8", [False, True])
@pytest.mark.parametrize("prefill,shape", [(False, (1, 1)), (False, (1, 3)), (False, (3, 1)), (True, (1, 5)), (True, (1, 1))])
def test_a_layer_takes_rows_in_more_than_two_dimensions(prefill, shape, int8):
    """A decoder layer flattens what comes in front of the hidden size, on one token and a few as on many."""
    from tinyllmforge_amd.config import ModelConfig
    from tinyllmforge_amd.layers.layernorm import RMSNorm
    from tinyllmforge_amd.models.qwen3 import Qwen3DecoderLayer
    from tinyllmforge_amd.utils.context import reset_context, set_context
    g, n, width, bs = torch.Generator(device=DEV).manual_seed(3), shape[0] * shape[1], 1024, 16
    cfg = ModelConfig(hidden_size=width, num_hidden_layers=1, num_attention_heads=16, num_key_value_heads=8, intermediate_size=512, vocab_size=16,
                      head_dim=128, max_position_embeddings=256)
    default = torch.get_default_dtype()
    torch.set_default_dtype(BF)
    try:
        with torch.device(DEV):
            layer, norm = Qwen3DecoderLayer(cfg).to(DEV), RMSNorm(width, EPS).to(DEV)
    finally:
        torch.set_default_dtype(default)
    for lin in (layer.self_attn.qkv_proj, layer.self_attn.o_proj, layer.mlp.gate_up_proj, layer.mlp.down_proj):
        rows, cols = lin.weight.shape
        if int8:
            lin.load_quantized(torch.randint(-127, 128, (rows, cols), dtype=torch.int8, device=DEV, generator=g), torch.full((rows,), cols ** -0.5 / 73, device=DEV))
            lin.finish_quantized_load()
            lin.pack_()
        else:
            lin.weight.data.normal_(0, cols ** -0.5, generator=g)
            if lin is layer.mlp.gate_up_proj:
                lin.interleave_()
    for m in (layer.self_attn.q_norm, layer.self_attn.k_norm, layer.post_attention_layernorm, norm):
        m.weight.data.fill_(1)
    attn = layer.self_attn.attn
    attn.k_cache, attn.v_cache = (torch.empty(2 * n, bs, 8, 128, dtype=BF, device=DEV).normal_(generator=g) for _ in range(2))
    i32 = lambda x: torch.tensor(x, dtype=torch.int32, device=DEV)
    if prefill:
        fields = dict(is_prefill=True, cu_seqlens_q=i32([0, n]), cu_seqlens_k=i32([0, n]), max_seqlen_q=n, max_seqlen_k=n, slot_mapping=i32(list(range(n))))
        positions = torch.arange(n, device=DEV)
    else:
        fields = dict(is_prefill=False, slot_mapping=i32([i * 32 + 20 for i in range(n)]), context_lens=i32([21] * n), block_tables=i32([[2 * i, 2 * i + 1] for i in range(n)]))
        positions = torch.full((n,), 20, device=DEV)
    x, residual = (torch.empty(n, width, dtype=BF, device=DEV).normal_(generator=g) for _ in range(2))
    outs = []
    for view in ((n, width), (*shape, width)):
        set_context(**fields)
        with torch.inference_mode():
            outs.append(layer.forward_normed(positions, x.view(view), residual.view(view), norm))
        reset_context()
    for a, b in zip(*outs):
        assert torch.equal(a, b.view(a.shape))
