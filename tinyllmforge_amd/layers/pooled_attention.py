"""Sigmoid attention over a sliding window and pooled blocks, on paged caches.

Position ``i`` sees the ``window`` tokens up to itself and one mean key / value per block of ``pool`` tokens that lies
wholly before them.  The layer owns two paged caches with common page numbers: token rows and block means."""
import torch
from torch import nn

from .. import ops
from ..utils.context import get_context


class PooledWindowAttention(nn.Module):
    def __init__(self, num_heads: int, num_kv_heads: int, head_dim: int, scale: float, window: int, pool: int,
                 rot_dims: int, rope: torch.Tensor, eps: float, dtype: torch.dtype):
        super().__init__()
        self.num_heads, self.num_kv_heads, self.head_dim = num_heads, num_kv_heads, head_dim
        self.scale, self.window, self.pool, self.rot_dims, self.eps = scale, window, pool, rot_dims, eps
        self.dtype = dtype
        self.register_buffer("cos_sin", rope, persistent=False)
        self.score_bias = nn.Parameter(torch.zeros(num_heads))
        self.takes_partials = head_dim % 8 == 0 and rot_dims % 8 == 0    # the preparation may add up split projections
        self.kv = None                      # ops.PooledKV, bound by the model runner

    # -- what the model runner asks a layer with a paged cache
    def page_bytes(self, block_size: int) -> int:
        return ops.PooledKV.page_bytes(block_size, self.num_kv_heads, self.head_dim, self.pool,
                                       torch.empty(0, dtype=self.dtype).element_size())

    def bind_pages(self, pages: int, block_size: int, device):
        self.kv = ops.PooledKV(pages, block_size, self.num_kv_heads, self.head_dim, self.pool, self.window,
                               self.dtype, device) if pages else None

    def forward(self, proj: torch.Tensor, q_bias, k_bias, positions: torch.Tensor) -> torch.Tensor:
        """``proj``: rows ``[q | k | gate]`` -> ``[N, heads * head_dim]``, gated.  Partial sums of a projection (``ops.Deferred``) are added up by the
        separate preparation, so portions of 17 to 64 and 385 to 768 rows of width 4096 come that way.  (Projection and attention, us, with partial sums and with rows
        that are finished and read by the attention: 400 rows 63.9 and 59.6, 700 90.1 and 86.4, 64 behind 512 45.3 and 43.2; int8 65.1 and 62.5, 89.3 and 84.2,
        41.1 and 41.1.)"""
        ctx, kv = get_context(), self.kv
        n, single, bias = proj.shape[0], ctx.num_single, self.score_bias.data
        out = torch.empty(n, self.num_heads * self.head_dim, dtype=proj.dtype, device=proj.device)
        portions, projected = ctx.cu_seqlens_q.numel() - 1 - single if single < n else 0, False
        if portions and self._from_projection(n - single, portions, proj.dtype):
            if isinstance(proj, ops.Deferred) and proj.splits == 1:
                proj = proj.rows()
            projected = isinstance(proj, torch.Tensor) and ops.pooled_attention_projected(
                proj, q_bias, k_bias, positions, self.cos_sin, self.rot_dims, ctx.slot_mapping, bias, kv, ctx.block_tables, ctx.cu_seqlens_q,
                ctx.seq_starts, single, portions, ctx.max_portion, self.scale, self.eps, out)
            if projected and not single:
                return out
        q, gate = ops.attn_prep(proj, q_bias, k_bias, positions, self.cos_sin, self.rot_dims, ctx.slot_mapping, kv.k,
                                kv.v, self.num_heads, self.head_dim, self.eps, rows=single if projected else None)
        if single:
            ops.pooled_attention_rows(q if projected else q[:single], bias, gate if projected else gate[:single], kv, ctx.block_tables,
                                      positions[:single], ctx.slot_mapping[:single], self.scale, ctx.max_len, out[:single], pool_new=True)
        if portions and not projected:
            ops.pool_blocks(kv, ctx.block_tables, ctx.cu_seqlens_q, ctx.seq_starts, single, portions, ctx.max_portion)
            if proj.dtype == torch.bfloat16:
                ops.pooled_attention_prefill(q, bias, gate, kv, ctx.block_tables, ctx.cu_seqlens_q, ctx.seq_starts,
                                             single, portions, ctx.max_portion, self.scale, out)
            else:
                ops.pooled_attention_rows(q[single:], bias, gate[single:], kv, ctx.block_tables, positions[single:],
                                          ctx.slot_mapping[single:], self.scale, ctx.max_len, out[single:],
                                          row_seq=ctx.row_seq[single:])
        return out

    def _from_projection(self, rows: int, portions: int, dtype) -> bool:
        """Whether portions make their queries where the attention reads them.  A workgroup makes those of a tile of rows, there or not, so many short
        portions are faster with rows prepared, the more so without a context.  us prepared and from the projection, 16 heads on 8, tiles of 64: 256 of up to 12 tokens
        22.1 and 29.2, of up to 35 34.4 and 37.3, 172 of up to 63 36.5 and 32.8; while they do not fill the chip the launches count: 64 of up to 20
        20.0 and 12.6, 128 of up to 35 23.8 and 22.4.  On the wrong side of it: 256 of up to 35 in tiles of 32, some in two of them, 44.3 and 45.9; 100 of up to 12 behind 256 held
        tokens 26.8 and 29.0; prepared, 256 of up to 26 in tiles of 64 behind 256 71.6 and 64.0."""
        if dtype != torch.bfloat16:
            return False
        tile = max(1, 128 * self.num_kv_heads // self.num_heads)
        return portions * self.num_kv_heads <= 1024 or rows * 7 >= portions * tile * 4
