"""Causal grouped-query attention whose heads mix their weights after the softmax, on paged head-major caches.

In front of it: RMS norm over the whole query and the whole key projection, rotation of neighbouring dimensions, a temperature
per head."""
import torch
from torch import nn

from .. import ops
from ..utils.context import get_context


def short_in_tiles(portions: int, rows: int, keys: int) -> bool:
    """Whether short portions, ``rows`` rows in all and contexts of up to ``keys``, go in row tiles: where they are few rows, row by row is faster.
    A row tile starts with more latency, and its keys are read once for all its rows: a row costs what it reads, a tile about as much as one row and
    all of them together as much as 40.  16 heads, the layer by rows and in tiles, us: portions behind 1024 keys, 8 of up to 8 tokens 57 and 67, 33 of 2
    74 and 94, 16 of 4 63 and 75, one of 64 63 and 62, 8 of up to 16 93 and 67, 60 of up to 32 818 and 135; behind 2048, 33 of 2 121 and 149, 12 of 6
    111 and 101, 100 of 2 326 and 310; behind 64, where either waits for the host, 33 of 2 41 and 37."""
    return rows >= 64 and (keys <= 256 or rows >= 55 + 1.1 * portions)


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
        short = 0 if short_in_tiles(ctx.num_short, ctx.num_short_rows - ctx.num_single, ctx.block_tables.stride(0) * kv.k.shape[2]) else ctx.num_short
        rows = (ctx.num_short_rows if short else ctx.num_single) if tiles else n
        if rows:
            ops.talk_attention_rows(q[:rows], kv, ctx.block_tables, positions[:rows], ctx.slot_mapping[:rows], self.talk.data, ctx.max_len,
                                    out[:rows], ctx.row_seq[:rows] if ctx.num_single < rows else None)
        if rows < n:
            first = ctx.num_single + short
            portions = ctx.cu_seqlens_q.numel() - 1 - first
            calls = [(first, portions, ctx.max_portion, n - rows)]
            if 0 < ctx.num_short - short < portions and not self._together(portions, n - rows):
                many, most = ctx.num_short, ctx.num_short_rows - rows
                calls = [(first, many, ctx.max_short, most), (first + many, portions - many, ctx.max_portion, n - rows - most)]
            for call in calls:
                ops.talk_attention_prefill(q, kv, ctx.block_tables, ctx.cu_seqlens_q, ctx.seq_starts, *call[:3], self.talk.data, out, call[3])
        return out

    def _together(self, portions: int, rows: int) -> bool:
        """Whether short and long portions share a call, which has workgroups for the row tiles of the longest in every portion: while these
        all fit the chip, or are cut, that is cheaper than two calls, the layer 65 us and 102 (16 heads, 3 of 300 tokens and 10 of 100).  Beyond
        that the empty ones take their turn: one of 8000 tokens and 200 of 2 took 9690 us together, 863 apart, one of 200 and 30 of 20 behind 1024 keys 215
        and 131, behind 64 63 and 89."""
        ctx = get_context()
        most = -(-ctx.max_portion // ops.talk_tile_rows(self.num_heads, self.num_kv_heads, self.dim, self.value_dim)) * portions
        keys = ctx.block_tables.stride(0) * self.kv.k.shape[2]
        return most <= 192 or (most <= 512 and keys <= 512) or ops.talk_prefill_cuts(self.kv, ctx.block_tables, portions, ctx.max_portion, rows, self.num_heads)
