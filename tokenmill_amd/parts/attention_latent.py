"""Attention through a shared latent.

Queries come from a narrow latent (down projection, RMS norm, up projection) and are laid out head by head as
[Dn channels without rotation | Dr rotated channels]. Keys and values come from one latent of Lk channels per token
(down projection, RMS norm) plus Dr rotated key channels that all heads share; head h's key is W_uk[h] c, its value
W_uv[h] c. Only the latent and the shared rotated channels are cached: one row of Lk + Dr numbers per token,
whatever the number of heads. The per-head matrices move to the other side of the two sums,

    score(t, j, h) = scale * ((W_uk[h]^T q_n[t, h]) . c_j + q_r[t, h] . k_r[j])
    out(t, h)      = W_uv[h] (sum_j softmax_j(score) c_j)

so that every head reads the same cached rows (a query of Lk + Dr channels, a result of Lk channels), in a prompt and
in decoding alike. Softmax over the visible rows: the token's own and the ``window - 1`` before it (None: all).
What a model may add, each a constructor parameter: a sigmoid gate per head computed from the mixer's input; a sink per
head (a learned number whose exponential joins the softmax's denominator, with no row behind it); a rotation of
neighbouring pairs or of pairs half the rotated width apart; no latent of its own (``own_kv`` False: the mixer reads
the rows that another layer caches, with its own queries and per-head matrices).
"""
from __future__ import annotations

import torch

from tokenmill_amd import profiling
from tokenmill_amd.hip import ops
from tokenmill_amd.parts.base import KVCacheSpec, KVCacheView, Mixer, StepContext, as_tensor, portion_blocks, portion_rows, portion_tiles
from tokenmill_amd.parts.linear import Linear
from tokenmill_amd.parts.position import RotaryEmbedding
from tokenmill_amd.weights.loader import TensorSpec


# A portion runs with keys and values per head where one of its tokens sees at least so many rows, up to so many of its own; portions pass
# together while their rows are no more. A (query, row) pair costs a third of what it costs over the latent, and a token's rows are walked by two
# wavefronts side by side; it is two launches more and one for each further portion, which short prompts have no use for. Beyond, keys and values would be no passing
# buffer any more (8,192 rows of the 2k shapes: 70 MB). Whole steps of the 2k Lusolix shape, onto the latent / by heads, us: prompts of 100 / 250 /
# 400 / 800 / 1,500 tokens 2,470 / 2,483 / 2,682 / 3,377 / 4,268 and 2,597 / 2,576 / 2,638 / 2,607 / 3,005 (up to 2,600 the launches are the
# time). The number of tokens decides nothing: a portion of up to 16 is one tile, four blocks, over the latent, that walk its rows one
# after the other. The mixer of one layer without a window, GPU time, us, 2 / 16 / 64 / 256 tokens behind 500, 1,000, 4,000 and 7,900 cached ones: over the
# latent 105 / 124 / 148 / 180, 179 / 193 / 221 / 253, 611 / 622 / 644 / 675, 1,164 / 1,180 / 1,199 / 1,232; by heads 46 / 56 / 65 / 70, 56 /
# 61 / 77 / 81, 119 / 124 / 133 / 141, 196 / 201 / 210 / 212. Portions in one step, 1 / 4 / 7 / 24: of 500 tokens 146 / 270 / 417 / 1,214 and 65 / 113 /
# 174 / 548; of 2 tokens behind 4,000 614 / 620 / 622 / 642 and 118 / 261 / 481 / 1,437. (Many of the last kind would be better off over the latent,
# but a step of the scheduler holds one request that goes on inside its prompt, and the choice is to hang on a portion alone.)
HEADS_SEEN_ROWS = 384
HEADS_MOST_ROWS = 8192


class LatentAttention(Mixer):
    def __init__(self, hidden: int, num_heads: int, head_dim: int, rot_dim: int, v_head_dim: int, q_rank: int, kv_rank: int,
                 scale: float, norm_eps: float, rotary: RotaryEmbedding | None = None, window: int | None = None,
                 output_gate: bool = True, sink: bool = False, own_kv: bool = True,
                 names: tuple[str, ...] = ("dq", "uq", "dkv", "uk", "uv", "g", "o"),
                 norm_names: tuple[str, str] = ("dq.norm", "dkv.norm"), suffixes: tuple[str, str] = ("", ".b"),
                 sink_name: str = "sink"):
        """``head_dim``: channels of a head's query and key that are not rotated; ``rot_dim``: the rotated ones (the key's are
        shared by the heads). ``rotary``: a ``RotaryEmbedding`` over ``rot_dim`` channels, of which it may rotate fewer, in
        either pairing; None: none. ``output_gate``: whether a per-head sigmoid gate (a projection of the input) multiplies the
        result. ``sink``: whether the checkpoint holds a number per head that joins the softmax's denominator. ``own_kv``
        False: no down projection to the key/value latent; the cache is another layer's."""
        if min(num_heads, head_dim, v_head_dim, q_rank, kv_rank) <= 0 or rot_dim < 0:
            raise ValueError("the sizes of a latent attention are positive")
        if kv_rank > ops.LATENT_MAX_RANK or kv_rank + rot_dim > ops.LATENT_MAX_ROW:
            raise ValueError(f"a latent of {kv_rank} + {rot_dim} channels: the kernels take {ops.LATENT_MAX_RANK} and rows of {ops.LATENT_MAX_ROW}")
        if rotary is not None and rotary.rotary_dim > rot_dim:
            raise ValueError("the rotation fits the rotated part of a head")
        if window is not None and window < 1:
            raise ValueError("a window holds at least one position")
        self.hidden, self.num_heads, self.head_dim, self.rot_dim, self.v_head_dim = hidden, num_heads, head_dim, rot_dim, v_head_dim
        self.q_rank, self.kv_rank, self.scale, self.norm_eps = q_rank, kv_rank, float(scale), float(norm_eps)
        self.rotary, self.window, self.output_gate = rotary, window, output_gate
        self.has_sink, self.own_kv, self.sink_name = sink, own_kv, sink_name
        self.half_pairs = rotary is not None and not rotary.interleaved
        self.row = kv_rank + rot_dim                                       # what a token caches
        n = dict(zip(("dq", "uq", "dkv", "uk", "uv", "g", "o"), names))
        self.names, self.norm_names, self.suffixes = n, norm_names, suffixes
        # the projections that read the mixer's input are one product: [query latent | latent | shared key | gates]
        outs, stacked = [q_rank], [n["dq"]]
        if own_kv:
            outs.append(kv_rank + rot_dim)
            stacked.append(n["dkv"])
        self.gate_at = sum(outs)
        if output_gate:
            outs.append(num_heads)
            stacked.append(n["g"])
        self.down = Linear(hidden, outs, stacked, bias=False, suffixes=suffixes)
        self.uq = Linear(q_rank, num_heads * (head_dim + rot_dim), n["uq"], bias=False, suffixes=suffixes)
        self.o = Linear(num_heads * v_head_dim, hidden, n["o"], bias=False, suffixes=suffixes)
        self.q_norm: torch.Tensor | None = None
        self.kv_norm: torch.Tensor | None = None
        self.sink: torch.Tensor | None = None           # float32 [H]
        self.uk: torch.Tensor | None = None             # [H, Dn, Lk]: a head's query channels onto the latent
        self.uv: torch.Tensor | None = None             # [H, Lk, Dv]: the latent onto a head's value channels
        self.uk_nt: torch.Tensor | None = None          # the same two as [H, N, K], the order the matrix-unit products read
        self.uv_nt: torch.Tensor | None = None

    def tensor_specs(self, prefix: str):
        H, Dn, Dv, Lk = self.num_heads, self.head_dim, self.v_head_dim, self.kv_rank
        sw = self.suffixes[0]
        specs = {**self.down.tensor_specs(prefix), **self.uq.tensor_specs(prefix), **self.o.tensor_specs(prefix)}
        specs[prefix + self.names["uk"] + sw] = TensorSpec((H * Dn, Lk))
        specs[prefix + self.names["uv"] + sw] = TensorSpec((H * Dv, Lk))
        specs[prefix + self.norm_names[0]] = TensorSpec((self.q_rank,), init="ones")
        if self.own_kv:
            specs[prefix + self.norm_names[1]] = TensorSpec((Lk,), init="ones")
        if self.has_sink:
            specs[prefix + self.sink_name] = TensorSpec((H,))
        return specs

    def load(self, tensors, prefix: str) -> None:
        H, Dn, Dv, Lk = self.num_heads, self.head_dim, self.v_head_dim, self.kv_rank
        sw = self.suffixes[0]
        self.down.load(tensors, prefix)
        self.uq.load(tensors, prefix)
        self.o.load(tensors, prefix)
        self.uk = tensors[prefix + self.names["uk"] + sw].view(H, Dn, Lk).contiguous()
        self.uv_nt = tensors[prefix + self.names["uv"] + sw].view(H, Dv, Lk)
        self.uv = self.uv_nt.transpose(1, 2).contiguous()
        self.uk_nt = self.uk.transpose(1, 2).contiguous() if self.uk.dtype == torch.bfloat16 else None
        # the norm weights meet 32-bit statistics and are kept in 32-bit
        self.q_norm = tensors[prefix + self.norm_names[0]].float().contiguous()
        self.kv_norm = tensors[prefix + self.norm_names[1]].float().contiguous() if self.own_kv else None
        self.sink = tensors[prefix + self.sink_name].float().contiguous() if self.has_sink else None
        if self.rotary is not None:
            self.rotary.load(tensors, prefix)

    def prepare(self, pack_weights: bool) -> None:
        for lin in (self.down, self.uq, self.o):
            lin.prepare(pack_weights)

    def cache_spec(self):
        return KVCacheSpec(1, self.row, self.window, values=False)

    def other_matrices(self) -> list[torch.Tensor]:
        """The matrices kept outside ``Linear`` parts (for a count of parameters)."""
        return [self.uk, self.uv]

    def visible_pairs(self, step: StepContext) -> tuple[int, int]:
        """(rows read, (query, row) pairs) of a step, for a profile's floor."""
        rows = pairs = 0
        for start, n in zip(step.start_positions, step.q_lens):
            first = max(0, start - self.window + 1) if self.window else 0
            rows += start + n - first
            for p in range(start, start + n):
                pairs += min(p + 1, self.window) if self.window else p + 1
        return rows, pairs

    def cost(self, label: str, step: StepContext | None, rows: int) -> tuple[int, int]:
        e = self.uq.weight.element_size()
        H, Dn, Dr, Dv, Lk = self.num_heads, self.head_dim, self.rot_dim, self.v_head_dim, self.kv_rank
        if label == "qkv":          # both down projections, the queries' up projection and their move onto the latent
            a, b = self.down.cost(rows, out_bytes=4), self.uq.cost(rows)
            return a[0] + b[0] + self.uk.numel() * e + rows * H * self.row * e, a[1] + b[1] + 2 * rows * H * Dn * Lk
        if label == "o_proj":       # the latent results onto the heads' values, and the output projection
            a = self.o.cost(rows)
            return a[0] + self.uv.numel() * e + rows * H * Lk * e, a[1] + 2 * rows * H * Lk * Dv
        seen, pairs = self.visible_pairs(step)
        return seen * self.row * e + step.num_tokens * H * (self.row + Lk) * e, 2 * pairs * H * (self.row + Lk)

    def _by_heads(self, q, step: StepContext) -> list[tuple[int, ...]]:
        """Which of the step's portions run with keys and values per head, made from their visible rows, in place of queries and results
        moved onto the latent: groups of requests whose rows fit the passing buffer together. A portion's own tokens and rows decide,
        never its neighbours'."""
        H, Dn, Lk, window = self.num_heads, self.head_dim, self.kv_rank, self.window or 0
        if not step.portions_known or step.num_decode >= q.shape[0] or q.dtype != torch.bfloat16 or self.uk_nt is None \
                or Lk % 64 or Lk < 256 or H * Dn % 8 or not ops.attn_heads_takes(Dn, self.rot_dim, self.v_head_dim):
            return []
        groups, held = [], HEADS_MOST_ROWS
        for s, (_, n, start, _, rows) in enumerate(portion_rows(step, window)):
            if min(start + n, window or start + n) < HEADS_SEEN_ROWS or rows > HEADS_MOST_ROWS:
                continue
            if held + rows > HEADS_MOST_ROWS:
                groups.append(())
                held = 0
            groups[-1] += (s,)
            held += rows
        return groups

    def _attend_by_heads(self, q, out, gate, step: StepContext, cache: KVCacheView, group, cos, sin, which: tuple[int, ...]) -> None:
        """The rows of ``out`` [T, H Dv] of the portions ``which``, gated."""
        H, Dn, Dr, Dv, Lk = self.num_heads, self.head_dim, self.rot_dim, self.v_head_dim, self.kv_rank
        blocks, gathers, rows = portion_blocks(step, which, self.window or 0, q.device)
        portions, bf16 = portion_rows(step, self.window or 0), dict(dtype=torch.bfloat16, device=q.device)
        span = slice(portions[which[0]][0], portions[which[-1]][0] + portions[which[-1]][1])       # (rows of other portions between: left alone)
        latent, kv = torch.empty((rows, Lk), **bf16), torch.empty(rows * (H * Dn + Dr), **bf16)
        keys, shared = kv[:rows * H * Dn].view(rows, H * Dn), kv[rows * H * Dn:].view(rows, Dr)
        vt, qr = torch.empty((H * Dv, rows), **bf16), torch.empty((span.stop - span.start, H * Dr), **bf16)
        for s, first, count, lo, hi, at in gathers:
            ops.latent_rows(cache.k, group.block_tables[s], first, lo, hi, Lk, Dr, latent[at:at + count], shared[at:at + count])
        ops.tile_linear(latent, self.uk.view(H * Dn, Lk), keys)
        ops.tile_linear(self.uv_nt.view(H * Dv, Lk), latent, vt)
        ops.rotate_heads(q[span, Dn:], Dn + Dr, qr, Dr, H, Dr, cos, sin, step.positions[span], half_pairs=self.half_pairs)
        ops.attn_heads(q[span], qr, kv, vt, out[span], blocks, H, Dn, Dr, Dv, self.scale, self.window or 0,
                       gate=gate[span] if gate is not None else None, sink=self.sink)

    @staticmethod
    def _latent_runs(step: StepContext, T: int, groups) -> list[tuple[int, int, tuple[int, ...] | None]]:
        """Runs of rows that no group holds: (first row, row behind the last, their portions' requests, None: the whole step's)."""
        if not groups:
            return [(0, T, None)]
        taken = {s for which in groups for s in which}
        runs = []
        for s, (row, n, _, _, _) in enumerate(portion_rows(step, 0)):
            if s in taken:
                continue
            if runs and runs[-1][1] == row:
                runs[-1] = (runs[-1][0], row + n, runs[-1][2] + (s,))
            else:
                runs.append((row, row + n, (s,)))
        if step.num_decode:
            first = T - step.num_decode
            if runs and runs[-1][1] == first:
                runs[-1] = (runs[-1][0], T, runs[-1][2])
            else:
                runs.append((first, T, ()))
        return runs

    def _attend(self, qa, latent, first: int, tiles, singles: int, step: StepContext, cache: KVCacheView, group) -> None:
        """Prompt portions (``tiles``) and ``singles`` single tokens behind them, rows ``first`` and up of the step, on the matrix unit
        where its kernel takes the sizes; the 32-bit path and every other size through the kernel that takes a token and a head a
        wavefront."""
        H, Lk, row, n = self.num_heads, self.kv_rank, self.row, qa.shape[0]
        seq, positions = step.seq_of_token[first:first + n], step.positions[first:first + n]
        if not ops.attn_latent_mfma_takes(qa.dtype, Lk, row, H) or (n > singles and (tiles is None or not tiles.shape[0])):
            ops.attn_latent(qa, latent, cache.k, group.block_tables, seq, positions, H, Lk, row, self.scale, self.window or 0, sink=self.sink)
            return
        if n > singles:
            ops.attn_latent_mfma(qa, latent, cache.k, group.block_tables, tiles, seq, positions, 0, 0, H, Lk, row, self.scale,
                                 self.window or 0, sink=self.sink)
        if singles > 0:
            ops.attn_latent_mfma(qa, latent, cache.k, group.block_tables, None, seq, positions, n - singles, singles, H, Lk, row, self.scale,
                                 self.window or 0, most_context=step.max_decode_context,
                                 bound=self.rotary.max_positions if self.rotary is not None else 1 << 20, sink=self.sink)

    def forward(self, x, step: StepContext, cache: KVCacheView, residual: torch.Tensor | None = None):
        x = as_tensor(x)
        T = x.shape[0]
        H, Dn, Dr, Dv, Lq, Lk, row = self.num_heads, self.head_dim, self.rot_dim, self.v_head_dim, self.q_rank, self.kv_rank, self.row
        rot = self.rotary
        if rot is not None and step.max_context_len > rot.max_positions:
            raise ValueError(f"position {step.max_context_len - 1} is beyond the rotary table ({rot.max_positions} positions)")
        cos, sin = (rot.cos, rot.sin) if rot is not None else (None, None)
        if cache.write != self.own_kv:
            raise ValueError("a mixer with a latent of its own writes its cache, one without reads another's: the model's run list disagrees")
        group = step.groups[cache.group]
        half = self.half_pairs
        with profiling.label("qkv", lambda: self.cost("qkv", step, T)):
            low = self.down.forward(x, out_dtype=torch.float32)                         # 32-bit: it feeds norms and the rotation
            cq = torch.empty((T, Lq), dtype=x.dtype, device=x.device)
            if self.own_kv:
                ops.latent_prepare(low, Lq, Lk, Dr, self.q_norm, self.kv_norm, self.norm_eps, cos, sin, step.positions,
                                   group.slot_mapping, cq, cache.k, half_pairs=half)
            else:
                ops.latent_prepare(low, Lq, 0, 0, self.q_norm, None, self.norm_eps, None, None, None, None, cq, None)
            q = self.uq.forward(cq)
        gate = low[:, self.gate_at:] if self.output_gate else None
        out = torch.empty((T, H * Dv), dtype=x.dtype, device=x.device)
        groups = self._by_heads(q, step)
        cost = lambda: self.cost("attention", step, T)              # (the whole step's: counted with the first piece)
        for which in groups:
            with profiling.label("attention", cost):
                self._attend_by_heads(q, out, gate, step, cache, group, cos, sin, which)
            cost = None
        for first, stop, which in self._latent_runs(step, T, groups):
            self._onto_latent(q, out, gate, step, cache, group, cos, sin, first, stop, which, cost)
            cost = None
        with profiling.label("o_proj", lambda: self.cost("o_proj", step, T)):
            return self.o.forward(out)

    def _onto_latent(self, q, out, gate, step: StepContext, cache: KVCacheView, group, cos, sin, first: int, stop: int, which, cost) -> None:
        """Rows first .. stop - 1 of ``out``, gated: the queries moved onto the latent, the attention over it, its result onto the values.
        ``which``: the requests whose portions they are, beside single tokens (None: the whole step). ``cost``: the attention's, for a
        profile, or None; the two products' are counted by the caller."""
        n, T, H, Dn, Dr, Dv, Lk, row = stop - first, q.shape[0], self.num_heads, self.head_dim, self.rot_dim, self.v_head_dim, self.kv_rank, self.row
        half = self.half_pairs
        qa = torch.empty((n, H * row), dtype=q.dtype, device=q.device)
        latent = torch.empty((n, H * Lk), dtype=q.dtype, device=q.device)
        q, out, positions = q[first:stop], out[first:stop], step.positions[first:stop]
        with profiling.label("qkv"):
            if self.uk_nt is not None and ops.heads_matmul_mfma_takes(q, Dn + Dr, self.uk_nt):
                # the heads' rotated channels go beside their part on the latent in the same launch
                ops.heads_matmul_mfma(q, Dn + Dr, self.uk_nt, qa, row, tail=Dr, cos=cos, sin=sin, positions=positions, half_pairs=half)
            else:
                ops.heads_matmul(q, Dn + Dr, self.uk, qa, row)
                if Dr:
                    ops.rotate_heads(q[:, Dn:], Dn + Dr, qa[:, Lk:], row, H, Dr, cos, sin, positions, half_pairs=half)
        with profiling.label("attention", cost):
            tiles = step.prefill_tiles if which is None else portion_tiles(step, which, q.device) if which else None
            self._attend(qa, latent, first, tiles, max(0, stop - (T - step.num_decode)), step, cache, group)
        with profiling.label("o_proj"):
            gate = gate[first:stop] if gate is not None else None
            if ops.heads_matmul_mfma_takes(latent, Lk, self.uv_nt):
                ops.heads_matmul_mfma(latent, Lk, self.uv_nt, out, Dv, gate=gate)
            else:
                ops.heads_matmul(latent, Lk, self.uv, out, Dv, gate=gate)
