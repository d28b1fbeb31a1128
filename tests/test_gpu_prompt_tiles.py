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
    out = torch.empty(q.shape)
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
