"""Prompt attention over batches whose planes and row tiles do not come out even: every row of every head is computed once, by the
workgroup that csrc/prompt_tiles.h names for it."""
import pytest
import torch

from tinyllmforge_amd import ops

pytestmark = pytest.mark.gpu
LENGTHS = [(1,), (33, 257), (700, 16, 129, 64, 5), (65,) * 9]


def plain(q, k, v):
    """``q [T, H, D]``, ``k, v [T, G, D]``: causal softmax attention in fp32, on the host."""
    q, k, v = q.float().cpu(), k.float().cpu(), v.float().cpu()
    T, H = q.shape[:2]
    out = torch.empty(T, H, v.shape[2])
    for h in range(H):
        s = q[:, h] @ k[:, h * k.shape[1] // H].T
        w = torch.softmax(s.masked_fill(torch.ones(T, T, dtype=torch.bool).triu(1), -torch.inf), dim=-1)
        out[:, h] = w @ v[:, h * k.shape[1] // H]
    return out


@pytest.mark.parametrize("lens", LENGTHS, ids=str)
@pytest.mark.parametrize("heads,kv_heads", [(2, 1), (6, 3), (12, 12), (16, 8)])
def test_every_row_of_uneven_batches(lens, heads, kv_heads):
    torch.manual_seed(1)
    dim, dev, BF = 128, "cuda", torch.bfloat16
    n, seqs = sum(lens), len(lens)
    q, k, v = (torch.randn(n, h, dim, device=dev).to(BF) for h in (heads, kv_heads, kv_heads))
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device=dev)
    want = torch.cat([plain(q[a:b].float() * dim ** -0.5, k[a:b], v[a:b]) for a, b in zip(cu.tolist(), cu.tolist()[1:])])
    # both outputs are bf16 of a result whose products enter with 11 or more significant bits: half an ulp, 2^-9, of the result,
    # and 2^-9 of the largest value for what the rounding of the operands adds
    close = lambda got: torch.testing.assert_close(got.float().cpu().view(want.shape), want, rtol=2 ** -8, atol=2 ** -8)

    close(ops.varlen_prefill_attention(q, k, v, cu, cu, max(lens), dim ** -0.5))

    kv = ops.SinkKV(sum(-(-m // 64) for m in lens), 64, kv_heads, dim, dim, BF, dev)
    tables = torch.full((seqs, max(-(-m // 64) for m in lens)), -1, dtype=torch.int32)
    page = 0
    for i, (a, m) in enumerate(zip(cu.tolist(), lens)):
        for j in range(0, m, 64):
            rows = min(64, m - j)
            tables[i, j // 64] = page
            kv.k[page, :, :rows] = k[a + j:a + j + rows].transpose(0, 1)
            kv.v[page, :, :rows] = v[a + j:a + j + rows].transpose(0, 1)
            page += 1
    scaled = (q.float() * (dim ** -0.5 * 1.4426950408889634)).to(BF)
    out = torch.full((n, heads * dim), torch.nan, device=dev, dtype=BF)
    ops.sink_attention_prefill(scaled, kv, tables.to(dev), cu, torch.zeros(seqs, dtype=torch.int32, device=dev), 0, seqs, max(lens), None, None,
                               None, out)
    want = torch.cat([plain(scaled[a:b].float() * 0.6931471805599453, k[a:b], v[a:b]) for a, b in zip(cu.tolist(), cu.tolist()[1:])])
    close(out)


@pytest.mark.parametrize("heads,kv_heads", [(1, 1), (8, 2), (12, 6)])
def test_halves_of_tiles_that_no_row_sees(heads, kv_heads):
    """Portions that end on either side of the halves of a tile, 32 keys, and row tiles of 128, 32 and 64 rows that do."""
    test_every_row_of_uneven_batches((31, 32, 33, 63, 64, 65, 95, 96, 97, 128, 160, 161, 226), heads, kv_heads)


@pytest.mark.parametrize("dim,vdim", [(32, 32), (56, 100), (96, 64), (128, 128), (136, 128), (128, 136)])
@pytest.mark.parametrize("cap", [None, 20.0, 50.0])
def test_weights_follow_a_growing_maximum(dim, vdim, cap):
    """Scores that climb by more than 2^8 at random keys, in even and odd halves of a tile, behind a prefix in the cache."""
    torch.manual_seed(dim + vdim)
    dev, BF, heads, start, new, log2e = "cuda", torch.bfloat16, 4, 70, 203, 1.4426950408889634
    total = start + new
    kv = ops.SinkKV(-(-total // 64), 64, 1, dim, vdim, BF, dev)
    k, v = torch.randn(total, dim) * 0.2, torch.randn(total, vdim)
    k[:, 0] = torch.cumsum((torch.rand(total) < 0.05).float() * torch.rand(total) * 30, 0)
    k, v = k.to(BF), v.to(BF)
    for j in range(0, total, 64):
        rows = min(64, total - j)
        kv.k[j // 64, 0, :rows, :dim], kv.v[j // 64, 0, :rows, :vdim] = k[j:j + rows].to(dev), v[j:j + rows].to(dev)
    q = torch.randn(new, heads, dim) * 0.3
    q[:, :, 0] = torch.tensor([1.0, -1.0, 0.0, 0.3])
    q = q.to(BF)
    padded = torch.zeros(new, heads, kv.k.shape[3], dtype=BF, device=dev)
    padded[..., :dim] = q.to(dev)
    out = torch.full((new, heads * vdim), torch.nan, device=dev, dtype=BF)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)
    ops.sink_attention_prefill(padded, kv, i32(*range(kv.k.shape[0])).view(1, -1), i32(0, new), i32(start), 0, 1, new, None, None, cap, out)
    s = torch.einsum("ihd,jd->hij", q.double(), k.double())             # scores in log 2 units, or 2 log2(e) / cap times them
    s = s / log2e if cap is None else cap * torch.tanh(s / log2e / 2)
    s = s.masked_fill(torch.arange(total) > torch.arange(start, total)[:, None], -torch.inf)
    want = torch.einsum("hij,jd->ihd", torch.softmax(s, -1), v.double())
    # bf16 result (2^-9) of weights with 16 significant bits and fp32 scores of up to 2^8
    torch.testing.assert_close(out.view(new, heads, vdim).double().cpu(), want, rtol=2 ** -8, atol=2 ** -10)


@pytest.mark.parametrize("vdim,offset,gap", [(128, 0, 8), (128, 4, 8), (120, 0, 4), (72, 8, 0), (68, 4, 0), (33, 0, 0), (64, 1, 3)])
def test_results_of_any_width_and_alignment(vdim, offset, gap):
    """Results leave a unit's two lanes 16 bytes at a time, 8 or 2, whatever rows and their start allow; the bits are the same."""
    torch.manual_seed(vdim)
    dev, BF, n, heads, dim = "cuda", torch.bfloat16, 77, 6, 64
    kv = ops.SinkKV(2, 64, 2, dim, vdim, BF, dev)
    kv.k.normal_()
    kv.v.normal_()
    q, gate = torch.randn(n, heads, dim, device=dev).to(BF), torch.randn(n, heads * vdim, device=dev).to(BF)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)
    def run(offset, gap):
        rows = torch.full((offset + n * (heads * vdim + gap),), 7.0, device=dev, dtype=BF)
        out = rows[offset:].view(n, heads * vdim + gap)[:, :heads * vdim]
        ops.sink_attention_prefill(q, kv, i32(1, 0).view(1, -1), i32(0, n), i32(0), 0, 1, n, None, gate, None, out)
        kept = rows.clone()
        kept[offset:].view(n, -1)[:, :heads * vdim] = 7.0
        assert (kept == 7).all()
        return out.clone()
    got = run(offset, gap)
    k, v = (t[[1, 0]].transpose(0, 1).flatten(1, 2)[:, :n].transpose(0, 1)[..., :w] for t, w in ((kv.k, dim), (kv.v, vdim)))
    want = plain(q.float() * 0.6931471805599453, k, v) * torch.sigmoid(gate.float().cpu().view(n, heads, vdim))
    torch.testing.assert_close(got.float().cpu().view(want.shape), want, rtol=2 ** -7, atol=2 ** -8)
    assert torch.equal(got, run(1, 5))


@pytest.mark.parametrize("lens", [(1,), (128,), (128, 5, 77), (100,) * 9, (129, 128, 3)], ids=str)
@pytest.mark.parametrize("dim,rot,vdim", [(64, 32, 64), (128, 64, 128)])
@pytest.mark.parametrize("heads", [3, 16])
def test_latent_portions_of_one_row_tile(lens, dim, rot, vdim, heads):
    """Up to 128 tokens the heads of a portion are dealt like row tiles."""
    torch.manual_seed(sum(lens))
    dev, BF, n = "cuda", torch.bfloat16, sum(lens)
    s = ops.LatentShape(heads, dim, rot, 64, vdim)
    q, turned = torch.randn(n, heads, dim + rot).to(BF), torch.randn(n, rot).to(BF)
    k, v = torch.randn(n, heads, dim).to(BF), torch.randn(n, heads, vdim).to(BF)
    latents = torch.zeros(n, s.lp, dtype=BF)
    latents[:, 64:64 + rot] = turned
    cu = torch.tensor([0, *torch.tensor(lens).cumsum(0)], dtype=torch.int32, device=dev)
    out = torch.full((n, heads * vdim), torch.nan, device=dev, dtype=BF)
    scale = (dim + rot) ** -0.5
    ops.latent_prefill(q.to(dev), torch.cat([k.flatten(1), v.flatten(1)], 1).to(dev), latents.to(dev), cu, torch.zeros_like(cu), cu, 0, len(lens), max(lens),
                       1 << 20, scale, s, out)
    keys = torch.cat([k, turned[:, None].expand(-1, heads, -1)], 2)
    want = torch.cat([plain(q[a:b].float() * scale, keys[a:b], v[a:b]) for a, b in zip(cu.tolist(), cu.tolist()[1:])])
    torch.testing.assert_close(out.float().cpu().view(want.shape), want, rtol=2 ** -8, atol=2 ** -8)


# A value that is infinite or no number belongs to the rows that see its key: weights of zero times it are no numbers.  Keys are taken in
# tiles of 64 and rows by waves of 32 (one head per KV head), and a wave computes no tile that none of its rows sees.
@pytest.mark.parametrize("dim,vdim", [(32, 32), (96, 64), (128, 128), (136, 128)])
@pytest.mark.parametrize("cap", [None, 20.0, 50.0])
def test_sinks_a_value_without_a_number_stays_in_its_tile(dim, vdim, cap):
    torch.manual_seed(dim)
    dev, BF, n = "cuda", torch.bfloat16, 200
    kv = ops.SinkKV(4, 64, 2, dim, vdim, BF, dev)
    kv.k.normal_()
    kv.v.normal_()
    q = torch.randn(n, 2, kv.k.shape[3], device=dev).mul(0.1).to(BF)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)
    def run():
        out = torch.full((n, 2 * vdim), 7.0, device=dev, dtype=BF)
        return ops.sink_attention_prefill(q, kv, i32(2, 0, 3, 1).view(1, -1), i32(0, n), i32(0), 0, 1, n, None, None, cap, out)
    want = run().clone()
    assert want.isfinite().all()
    for key, value in ((100, torch.nan), (127, torch.inf), (64, -torch.inf)):    # rows 0 .. 63: two waves of the same workgroup
        kept = kv.v[0, :, key - 64].clone()
        kv.v[0, :, key - 64] = value
        got = run()
        assert torch.equal(got[:64], want[:64]) and not got[key:].isfinite().any(), key
        kv.v[0, :, key - 64] = kept


@pytest.mark.parametrize("dim,rot,vdim", [(24, 8, 32), (64, 32, 64), (64, 64, 128), (128, 64, 128)])
def test_latent_a_value_without_a_number_stays_in_its_tile(dim, rot, vdim):
    torch.manual_seed(dim)
    dev, BF, n, heads = "cuda", torch.bfloat16, 300, 2
    s = ops.LatentShape(heads, dim, rot, 64, vdim)
    q, latents = torch.randn(n, heads, s.dq, device=dev).to(BF), torch.randn(n, s.lp, device=dev).to(BF)
    expanded = torch.randn(n, heads * (dim + vdim), device=dev).to(BF)
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)
    def run(window):
        out = torch.full((n, heads * vdim), 7.0, device=dev, dtype=BF)
        return ops.latent_prefill(q, expanded, latents, i32(0, n), i32(0), i32(0, n), 0, 1, n, window, 0.1, s, out)
    # rows 0 .. 63 do not see the tile of key 100.  With a window of 100 the tiles of rows 128 .. 255 begin at key 29, and the first one is
    # not seen by rows 224 .. 255; the second one, of key 100, is
    for window, key, kept in ((1 << 20, 100, [(0, 64)]), (100, 40, [(224, 300)]), (100, 80, [(224, 300)]), (100, 100, [(0, 64), (256, 300)])):
        want, held = run(window).clone(), expanded[key].clone()
        assert want.isfinite().all()
        expanded[key, heads * dim:] = torch.nan
        got = run(window)
        expanded[key] = held
        for a, b in kept:
            assert torch.equal(got[a:b], want[a:b]), (window, key, a)
        assert got[key:min(key + window, n)].isnan().all(), (window, key)


def test_latent_maxima_follow_where_one_of_the_wave_grows():
    """Every tile's first key is the largest so far: by 2^20 and more for every sixteenth row, by less than 2^8 for those between, whose
    maxima have to move for their own sake only in every second tile."""
    torch.manual_seed(3)
    dev, BF, n, heads, dim, vdim = "cuda", torch.bfloat16, 1024, 16, 64, 128
    s = ops.LatentShape(heads, dim, 8, 64, vdim)
    k, v = torch.zeros(n, heads, dim), torch.randn(n, heads, vdim).to(BF)
    k[:, :, 0] = -400.0
    k[::64, :, 0] = 20.0 * torch.arange(n // 64)[:, None]
    k[::64, :, 1] = 3 * torch.rand(n // 64, heads)
    k, q = k.to(BF), torch.zeros(n, heads, s.dq, dtype=BF)
    q[..., :2] = 0.3
    q[::16, :, :2] = 1
    i32 = lambda *x: torch.tensor(x, dtype=torch.int32, device=dev)
    out = torch.full((n, heads * vdim), 7.0, device=dev, dtype=BF)
    ops.latent_prefill(q.to(dev), torch.cat([k.flatten(1), v.flatten(1)], 1).to(dev), torch.zeros(n, s.lp, dtype=BF, device=dev), i32(0, n), i32(0),
                       i32(0, n), 0, 1, n, 1 << 20, 0.6931471805599453, s, out)
    scores = torch.einsum("ihd,jhd->hij", q[..., :2].double(), k[..., :2].double()) * torch.tensor(0.6931471805599453).double()
    w = torch.softmax(scores.masked_fill(torch.ones(n, n, dtype=torch.bool).triu(1), -torch.inf), -1)
    want = torch.stack([w[h] @ v[:, h].double() for h in range(heads)], 1)
    # the largest weight is 1, those behind it are below 2^-5 and off by 2^-18 of themselves on average: 2^-23 of the result, and as much for
    # the roundings of exponents and sums.  A result 2^-22 off misses its nearest value where it lies that close to the middle between two
    # of them, which are 2^-8 to 2^-7 of it apart: 2^-14 of the results at most.  Largest weights of 16 bits made 2^-12 of them miss
    assert (out.view(n, heads, vdim).cpu() != want.to(BF)).double().mean().item() < 2 ** -14


@pytest.mark.parametrize("heads,dim,rot,rank", [(16, 64, 32, 256), (32, 128, 64, 512), (3, 24, 8, 64), (5, 40, 24, 1000), (1, 32, 32, 8)])
@pytest.mark.parametrize("n", [1025, 1030, 2051])
def test_latent_rows_of_prompts_are_prepared_as_few_are(heads, dim, rot, rank, n):
    """Beyond 1024 rows of the plain form two tokens go to a workgroup; up to there, and of other forms, latents and queries have workgroups
    of their own.  Rows without a slot or a position among them, columns between queries and latents; the bits are the same."""
    torch.manual_seed(n + rank)
    dev, BF = "cuda", torch.bfloat16
    s, col = ops.LatentShape(heads, dim, rot, rank, 16), heads * (dim + rot) + 16
    proj, norm = torch.randn(n, col + rank + rot + 8, device=dev).to(BF), torch.randn(rank, device=dev).to(BF)
    angles = torch.rand(512, rot // 2, device=dev) * 6.3
    table = torch.cat([angles.cos(), angles.sin()], 1)
    positions, slots = torch.randint(0, 512, (n,), device=dev), torch.randperm(64 * 40, device=dev)[:n].to(torch.int32)
    positions[::97], positions[5::101], slots[3::53], slots[7::59] = -1, 512, -1, 64 * 40
    def run(parts):
        cache, q = torch.full((40, 64, s.lp), 7.0, device=dev, dtype=BF), []
        for a in range(0, n, parts):
            at = slice(a, min(n, a + parts))
            q.append(ops.latent_prep(proj[at], col, norm, positions[at], table, slots[at], cache, s, 1e-6))
        return torch.cat(q), cache
    (q, cache), (q0, cache0) = run(n), run(1024)
    assert torch.equal(q, q0) and torch.equal(cache, cache0)


def test_more_workgroups_than_a_dimension_of_a_launch_holds():
    """The longest portion is the caller's bound: 2000 short ones under a bound of 300000 tokens are 12.5 million workgroups."""
    torch.manual_seed(0)
    lens = torch.tensor([1 + i % 3 for i in range(2000)])
    n, dev, BF = int(lens.sum()), "cuda", torch.bfloat16
    q, k, v = (torch.randn(n, 8, 128, device=dev).to(BF) for _ in range(3))
    cu = torch.cat([torch.zeros(1, dtype=torch.int64), lens.cumsum(0)]).to(torch.int32).to(dev)
    want = ops.varlen_prefill_attention(q, k, v, cu, cu, 3, 128 ** -0.5)
    assert torch.equal(ops.varlen_prefill_attention(q, k, v, cu, cu, 300000, 128 ** -0.5), want)
