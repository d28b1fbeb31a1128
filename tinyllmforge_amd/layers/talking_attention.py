"""Causal grouped-query attention whose heads mix their weights after the softmax, on paged head-major caches.

In front of it: RMS norm over the whole query and the whole key projection, rotation of neighbouring dimensions, a temperature
per head."""
import torch
from torch import nn

from .. import ops
from ..utils.context import get_context


class TalkingHeadsAttention(nn.Module):
    def __init__(self, num_heads: int, num_kv_heads: int, dim: int, value_dim: int, scale: float, eps: float, dtype: torch.dtype,
                 rot_dims: int = 0, rope=None):
        super().__init__()
        self.num_heads, self.num_kv_heads, self.dim, self.value_dim = num_heads, num_kv_heads, dim, value_dim
        self.scale, self.eps, self.dtype, self.rot_dims = scale, eps, dtype, rot_dims
        self.register_buffer("cos_sin", rope, persistent=False)
        self.parts = {"q": num_heads * dim, "k": num_kv_heads * dim, "v": num_kv_heads * value_dim}
        self.q_norm, self.k_norm = nn.Module(), nn.Module()
        self.q_norm.weight, self.k_norm.weight = nn.Parameter(torch.ones(self.parts["q"])), nn.Parameter(torch.ones(self.parts["k"]))
        self.temp = nn.Parameter(torch.ones(num_heads))
        self.talk = nn.Parameter(torch.eye(num_heads))
        self.kv = None                      # ops.SinkKV, bound by the model runner

    # -- what the model runner asks a layer with a paged cache
    def page_bytes(self, block_size: int) -> int:
        return ops.SinkKV.page_bytes(block_size, self.num_kv_heads, self.dim, self.value_dim, self.dtype.itemsize)

    def bind_pages(self, pages: int, block_size: int, device):
        self.kv = ops.SinkKV(pages, block_size, self.num_kv_heads, self.dim, self.value_dim, self.dtype, device) if pages else None

    def forward(self, proj, positions: torch.Tensor) -> torch.Tensor:
        """``proj``: rows ``[q | k | v]`` -> ``[N, heads * value_dim]``."""
        ctx, kv, n = get_context(), self.kv, proj.shape[0]
        q = ops.talk_prep(proj, kv, self.num_heads, positions, ctx.slot_mapping, self.q_norm.weight.data, self.k_norm.weight.data,
                          self.temp.data, self.cos_sin, self.rot_dims, self.eps, self.scale)
        out = torch.empty(n, self.num_heads * self.value_dim, dtype=self.dtype, device=q.device)
        tiles = self.dtype == torch.bfloat16 and ops.talk_prefill_supported(self.num_heads, self.num_kv_heads, self.dim, self.value_dim)
        rows, calls = self._calls(n) if tiles else (n, ())
        if rows:
            ops.talk_attention_rows(q[:rows], kv, ctx.block_tables, positions[:rows], ctx.slot_mapping[:rows], self.talk.data, ctx.max_len,
                                    out[:rows], ctx.row_seq[:rows] if ctx.num_single < rows else None)
        for first, load in calls:
            ops.talk_attention_prefill(q, kv, ctx.block_tables, ctx.cu_seqlens_q, ctx.seq_starts, first, *load[:2], self.talk.data, out, *load[2:])
        return out

    def _calls(self, n: int):
        """Rows of the step that run row by row, and the calls in row tiles: the first sequence of each, and its portions, their most tokens, rows,
        reads and most keys.  The same for all layers of a step."""
        ctx = get_context()
        single, near = ctx.num_single, ctx.num_short_rows if ctx.num_short else ctx.num_single
        if single >= n or (near >= n and near - single < 64):
            return n, ()                                             # few rows, where the host is waited for: not even asked
        key = ("talk", self.num_heads, self.num_kv_heads, self.dim, self.value_dim, n)
        if key not in ctx.plans:
            first, seqs = single + ctx.num_short, ctx.cu_seqlens_q.numel() - 1
            short = (ctx.num_short, ctx.max_short or ctx.max_portion, near - single)
            long = (seqs - first, ctx.max_portion if seqs > first else 0, n - near)
            reads, most = ctx.portion_reads, ctx.block_tables.stride(0) * self.kv.k.shape[2]
            if reads is None:                                        # as if contexts were half as long as the table
                reads = (short[2] * most // 2, most, long[2] * most // 2, most)
            short, long = short + reads[:2], long + reads[2:]
            route = ops.talk_prefill_route(self.kv, self.num_heads, single, short, long) if near - single >= 64 else 0
            both = (short[0] + long[0], max(short[1], long[1]), short[2] + long[2], short[3] + long[3], max(short[4], long[4]))
            calls = ([(first, long)], [(single, both)], [(single, short), (first, long)])[route]
            ctx.plans[key] = near if route == 0 else single, [c for c in calls if c[1][0]]
        return ctx.plans[key]
