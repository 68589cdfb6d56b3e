"""Two mixers whose softmax has a sink -- one more summand exp(sink[head]) in the denominator, a learned number a
head that stands for no key and brings no value -- and whose queries see the keys that a mask rule names: the last
`size` positions (`window`; with `keep_first` the request's first tokens besides) or the positions of the query's own
block of `size` (`chunk`), counted from the request's first token.  Scores may be capped, c tanh(score / c).

`SinkAttention`: grouped-query attention with query/key and value sizes of their own, optional biases on q, k, v,
a norm per head of q and k before the rotation (or after it; with a weight shared by the heads or without one), a
rotation of a head's first channels (how many, their pairing and the angles are the position part's), and
optionally a gate on the heads' outputs (sigmoid(Wg x), before the output projection).  Per token the cache keeps
keys [kv_heads, head_dim] and values [kv_heads, value_dim], both row-major.  The sink may be left out: the usual
softmax.

`LatentAttention`: keys and values of all heads are up-projections of ONE normed latent vector a token, plus one
rotated key part that all heads share; only the latent vector and that part are cached, [rank + rot_dim] a token.
The up-projections are moved to the query's side: q_lat[h] = W_uk[h]^T q_plain[h], so a head's score is
q_lat[h] . latent + q_rot[h] . k_rot -- attention of all heads over ONE shared key row whose first `rank` channels
are also the value -- and the head's output is W_uv[h] applied to the attention's latent result.  With `q_rank` the
queries come through a normed latent of their own, q = W_uq norm(W_dq x).  With `head_gate` every head's output is
multiplied by ONE number, sigmoid(Wg x)[head], before the output projection.
"""
from __future__ import annotations

import torch

from ..cache.manager import PAGE, PagedSpec
from ..weights.loader import WeightSpec, stacked
from .registry import PartError, build_part, register_part


def _mask_of(spec):
    if spec.mask is None:
        return None, 0
    if spec.mask.kind not in ("window", "chunk") or spec.mask.size < 1:
        raise PartError(f"mask {spec.mask.kind!r} of size {spec.mask.size}: window or chunk, of a positive size")
    if spec.mask.keep_first < 0 or (spec.mask.keep_first > 0 and spec.mask.kind != "window"):
        raise PartError("a window may keep a request's first tokens")
    return spec.mask.kind, int(spec.mask.size)


def _rope_table(position, ctx, device, rot_limit):
    """(the position part's table, whether its pairs are interleaved), or (None, False) without a rotation."""
    if position is None:
        return None, False
    rotation = position.rotation(ctx.max_positions, device)
    if rotation is None:
        return None, False
    if rotation.dim % 2 != 0 or not 2 <= rotation.dim <= rot_limit or rotation.table.shape[1] != rotation.dim:
        raise PartError(f"the position part turns {rotation.dim} channels: must be even, at most {rot_limit}")
    return rotation.table, bool(rotation.interleaved)


# Prompt portions of a model with a router keep the 64-column kernel and, in latent attention, the queries moved into the
# latent space, in both of which the sums of a row are rounded as they always were.  The portion kernel and made keys are no
# less precise (against 64 bits the median row of 640 is off by 0.26 % either way) but round elsewhere, and then other tokens
# are the ones whose choice of experts lies within rounding: of 640 scored rows of 1777-token prompts 6 had another choice than
# 64 bits, with portions 8, with either of the two alone 5 and 6, and only some of them the same.  Such a row's logits differ
# by a third, so a prompt would be scored otherwise than before.  (That prompt in 8 layers of 2048 channels: 3.82 ms, with
# portions 2.47.)
#
# Portions of latent attention that make keys and values of their own: from this many tokens and keys on (16 heads, rank
# 512, a step of eight layers of which two are latent attention, made against moved: 32 tokens behind 1000 keys 1.92 ms
# against 2.02, behind 4000 2.10 against 3.01; without context 512 tokens 3.17 against 3.09, 2048 5.4 against 6.5), and up
# to this many keys (the scratch memory: 9.3 KB a key).  The line holds for other ranks and heads too, though a small rank
# spares products either way: eight latent layers, 32 tokens behind 768, 128 behind 872 and a prompt of 2048, made against
# moved, at rank 64 with 16 heads 0.98 and 0.98, 1.10 and 1.15, 1.30 and 1.98 ms; at rank 128 0.90 and 1.09, 1.04 and 1.26,
# 1.27 and 3.20; at rank 128 with 4 heads 0.93 and 1.03, 1.09 and 1.23, 1.18 and 2.07.  A step that is replayed as a graph
# keeps the moved queries (see `_portions`).
PORTION_ROWS = 32
PORTION_LEAST_KEYS = 768
PORTION_KEYS = 16384


def _portion_library(weight):
    return ["portion_attention"] if weight is not None and weight.dtype == torch.bfloat16 else []


def _row_ranges(segments, without):
    """The batch rows of the step's entries but those `without`, as few ranges as there are."""
    ranges = []
    for i, (_, row, n, _) in enumerate(segments):
        if i in without:
            continue
        if ranges and ranges[-1][1] == row:
            ranges[-1] = (ranges[-1][0], row + n)
        else:
            ranges.append((row, row + n))
    return ranges


PARTIAL_CAP = 8 << 20         # floats that the shares of the key ranges of one launch may take at most
RANGE_KEYS = 128              # the narrowest key range of a workgroup
MOST_RANGES = 16              # key ranges of a group at most


def _groups_plan(rows, q_heads, kv_heads, value_dim):
    """The token-group vectors and the room for key ranges' shares that `attend` asks the step's context for."""
    from ..kernels.ops import Kernels
    big_heads, big_tokens, _, small_tokens = Kernels.sink_tiles_layout(q_heads, kv_heads)
    factors = {max(1, big_tokens // small_tokens)} | {columns // min(big_heads, 32) // small_tokens for columns in (64, 128)}
    return {**{(f"token_groups_{small_tokens}_{factor}", torch.int32): 2 * rows + 2 for factor in sorted(factors)},
            ("sink_partial", torch.float32): min(PARTIAL_CAP, Kernels.sink_partial_numel(rows, small_tokens, q_heads, value_dim, MOST_RANGES))}


def _key_ranges(ctx, groups, tokens, workgroups, q_heads, value_dim, mask, mask_size, keep_first=0):
    """(keys a range, ranges, room for their shares) for a launch over `groups` groups of single tokens or short portions
    that has `workgroups` workgroups without ranges: where those do not fill the GPU, a group's keys (its window or
    chunk; without a mask the step's longest context) are dealt out to several workgroups, as many as reach twice
    `target_workgroups` (four a compute unit), none narrower than RANGE_KEYS, and no more than their shares have room for.
    Single tokens of requests of 100 to 1200 keys, Sagopel's sizes: 48 of them 1741 us a step for 1762 with half as many
    workgroups, 128 2699 for 2790; Pamunex's latent attention 1393 for 1420 and 1946 for 2064; three times as many: 1755,
    2681, 1387, 1894.  Batches of 16 or less, which RANGE_KEYS and MOST_RANGES bound, take the same."""
    k = ctx.kernels
    reach = (mask_size if mask == "chunk" else mask_size + tokens - 1) if mask is not None else ctx.max_context
    if mask is not None and keep_first > 0:
        reach += -(-keep_first // 32) * 32
    reach = min(reach, ctx.max_context + 31) + 31             # (ranges start at the first tile, which may start earlier)
    most = max(1, min(MOST_RANGES, -(-reach // RANGE_KEYS), -(-2 * ctx.target_workgroups // max(1, workgroups))))
    room = ctx.workspace.get("sink_partial", (min(PARTIAL_CAP, k.sink_partial_numel(groups, tokens, q_heads, value_dim, most)),),
                             torch.float32)
    most = min(most, room.numel() // k.sink_partial_numel(groups, tokens, q_heads, value_dim, 1))
    if most <= 1:
        return 0, 1, None
    keys = -(-(-(-reach // most)) // 32) * 32
    return keys, -(-reach // keys), room


def portion_columns(ctx, q_heads, least=128):
    """Columns (token, head) of a portion kernel's workgroup: 128 (half the staging a column of those of 64) when the step
    brings at least `least` columns for every compute unit: one such workgroup each, or, where a workgroup has its compute unit
    to itself and workgroups of 64 would take their turns, every second."""
    return 128 if ctx.n_tokens * q_heads >= least * ctx.compute_units else 64


def attend(ctx, q, k_pages, v_pages, view, sink, out, q_heads, kv_heads, key_dim, value_dim, scale, mask, mask_size,
           keep_first=0, softcap=None, without=(), rest="rest"):
    """Every token of the step over the keys it sees (but those of the entries `without`, see `token_groups`).  The bfloat16 engine on the
    matrix cores where they take the sizes (prompt portions in workgroups of 128 or 64 columns, single tokens and short
    portions in workgroups of 16 whose wavefronts share the value channels); else, and in the float engine, one wavefront
    a (token, head), whose sums follow from the token's position alone."""
    k = ctx.kernels
    if k.sink_tiles_supported(key_dim, value_dim, k_pages.shape[3], v_pages.shape[3], view.page_size, mask, mask_size,
                              ctx.max_positions, keep_first) and q.shape[1] % 8 == 0:
        big_heads, big_tokens, small_heads, small_tokens = k.sink_tiles_layout(q_heads, kv_heads)
        portions = not ctx.routed and k.portion_attention_supported(q_heads, kv_heads, key_dim, value_dim, k_pages.shape[3], v_pages.shape[3],
                                                                    view.page_size, mask, mask_size, ctx.max_positions, keep_first, scale)
        rows = not portions and k.sink_rows_supported(key_dim, value_dim, k_pages, v_pages, view.page_size, mask, mask_size,
                                                      ctx.max_positions, keep_first, (q, out))
        if portions or rows:
            columns, big_heads = portion_columns(ctx, q_heads, 64 if rows else 128), min(big_heads, 32)
            big_tokens = columns // big_heads
        small, big, _ = ctx.token_groups(small_tokens, max(1, big_tokens // small_tokens), without, rest)
        if portions and big[2] > 0:
            k.portion_attention(q, k_pages, v_pages, view.block_table, ctx.slots, ctx.positions, sink, out, *big, columns, big_heads,
                                q_heads, kv_heads, key_dim, value_dim, view.page_size, scale, mask, mask_size, ctx.max_positions,
                                keep_first, softcap)
            big = (None, None, 0)
        if rows and big[2] > 0:
            k.sink_attention_rows(q, k_pages, v_pages, view.block_table, ctx.slots, ctx.positions, sink, out, *big, big_heads, q_heads,
                                  kv_heads, key_dim, value_dim, view.page_size, scale, mask, mask_size, ctx.max_positions, keep_first,
                                  softcap)
            big = (None, None, 0)
        for (first, count, n), heads, split in ((big, big_heads, False), (small, small_heads, True)):
            if n == 0:
                continue
            keys, ranges, room = (0, 1, None)
            if split:
                per_group = kv_heads * -(-(q_heads // kv_heads) // heads)
                keys, ranges, room = _key_ranges(ctx, n, small_tokens, n * per_group, q_heads, value_dim, mask, mask_size,
                                                 keep_first)
            k.sink_attention_tiles(q, k_pages, v_pages, view.block_table, ctx.slots, ctx.positions, sink, out, first,
                                   count, n, heads, split, q_heads, kv_heads, key_dim, value_dim, view.page_size,
                                   scale, mask, mask_size, ctx.max_positions, partial=room, split_keys=keys, splits=ranges,
                                   keep_first=keep_first, softcap=softcap)
        return
    k.sink_attention(q, k_pages, v_pages, view.block_table, ctx.slots, ctx.positions, sink, out, q_heads, kv_heads,
                     key_dim, value_dim, view.page_size, scale, mask, mask_size, keep_first, softcap)


@register_part("mixer", "sink_attention")
class SinkAttention:
    graph_safe = True

    def __init__(self, spec):
        s = self.spec = spec
        if s.q_heads % s.kv_heads != 0:
            raise PartError(f"q_heads {s.q_heads} is no multiple of kv_heads {s.kv_heads}")
        self.mask, self.mask_size = _mask_of(s)
        self.keep_first = s.mask.keep_first if s.mask is not None else 0
        if s.softcap is not None and not s.softcap > 0:
            raise PartError("softcap must be positive")
        if s.qk_norm is not None and s.qk_norm.size != s.head_dim:
            raise PartError("the q/k norm must span one head")
        self.position = build_part("position", s.position) if s.position is not None else None
        self.q_width, self.k_width, self.v_width = s.q_heads * s.head_dim, s.kv_heads * s.head_dim, s.kv_heads * s.value_dim
        self.o_width = s.q_heads * s.value_dim
        if s.gate not in (None, "sigmoid", "silu"):
            raise PartError(f"gate {s.gate!r}: sigmoid, silu or none")
        self.norm_order = None if s.qk_norm is None else "after" if s.qk_norm_after_rotation else "before"
        self.out_name = "mixer_out"                      # (a part that runs several mixers gives each a buffer of its own)
        self.qkv = self.o = self.bias = self.q_norm = self.k_norm = self.sink = None

    def weight_specs(self):
        s = self.spec
        specs = {"q": WeightSpec((self.q_width, s.hidden), stack="qkv"), "k": WeightSpec((self.k_width, s.hidden), stack="qkv"),
                 "v": WeightSpec((self.v_width, s.hidden), stack="qkv"), "o": WeightSpec((s.hidden, self.o_width))}
        if s.gate is not None:                           # (behind q, k, v: one projection gives all four)
            specs["g"] = WeightSpec((self.o_width, s.hidden), stack="qkv")
        if s.bias:
            for name, width in (("q.b", self.q_width), ("k.b", self.k_width), ("v.b", self.v_width)):
                specs[name] = WeightSpec((width,), keep_float32=True, init=("normal", 0.0, 0.02))
        if s.qk_norm is not None and s.qk_norm_weight:
            specs["q.norm"] = WeightSpec((s.head_dim,), keep_float32=True)
            specs["k.norm"] = WeightSpec((s.head_dim,), keep_float32=True)
        if s.sink:
            specs["sink"] = WeightSpec((s.q_heads,), keep_float32=True, init=("normal", 0.0, 1.0))
        return specs

    def bind(self, weights):
        s = self.spec
        self.qkv = stacked([weights[n] for n in (("q", "k", "v", "g") if s.gate is not None else ("q", "k", "v"))])
        self.o = weights["o"]
        self.bias = torch.cat([weights["q.b"], weights["k.b"], weights["v.b"]]).contiguous() if s.bias else None
        if s.qk_norm is not None and s.qk_norm_weight:
            self.q_norm, self.k_norm = weights["q.norm"], weights["k.norm"]
        self.sink = weights["sink"] if s.sink else None

    def cache_spec(self):
        s = self.spec
        return PagedSpec((("k", (s.kv_heads, PAGE, s.head_dim)), ("v", (s.kv_heads, PAGE, s.value_dim))),
                         self.mask_size if self.mask is not None else None, keep_first=self.keep_first)

    def libraries(self):
        return ["gemm", "sink_attention", "elementwise"] + _portion_library(self.o)

    def workspace_plan(self, rows, dtype, limits):
        s = self.spec
        gate = self.o_width if s.gate is not None else 0
        return {("sink_proj", dtype): rows * (self.q_width + self.k_width + self.v_width + gate), ("q", dtype): rows * self.q_width,
                ("attn", dtype): rows * self.o_width, (self.out_name, dtype): rows * s.hidden,
                **_groups_plan(rows, s.q_heads, s.kv_heads, s.value_dim)}

    def forward(self, ctx, x, cache_id, write_cache=True):
        s = self.spec
        k = ctx.kernels
        m = x.shape[0]
        proj = ctx.workspace.get("sink_proj", (m, self.qkv.shape[0]), x.dtype)
        k.gemm(x, self.qkv, proj)
        view = ctx.cache.paged_view(cache_id)
        k_pages, v_pages = view.tensors["k"], view.tensors["v"]
        q = ctx.workspace.get("q", (m, self.q_width), x.dtype)
        rope, interleaved = _rope_table(self.position, ctx, x.device, s.head_dim)
        qkv_width = self.q_width + self.k_width + self.v_width
        k.sink_qkv_prep(proj, self.bias, q, k_pages, v_pages, view.block_table, ctx.slots, ctx.positions, self.q_norm,
                        self.k_norm, s.qk_norm.eps if s.qk_norm is not None else 0.0, rope, s.q_heads, s.kv_heads,
                        s.head_dim, s.value_dim, view.page_size, write_cache, norm=self.norm_order, interleaved=interleaved)
        attn = ctx.workspace.get("attn", (m, self.o_width), x.dtype)
        attend(ctx, q, k_pages, v_pages, view, self.sink, attn, s.q_heads, s.kv_heads, s.head_dim, s.value_dim,
               float(s.scale), self.mask, self.mask_size, self.keep_first, s.softcap)
        if s.gate is not None:
            k.gate_mul(attn, proj[:, qkv_width:], attn, s.gate)
        out = ctx.workspace.get(self.out_name, (m, s.hidden), x.dtype)
        k.gemm(attn, self.o, out)
        return out


@register_part("mixer", "latent_attention")
class LatentAttention:
    graph_safe = True

    def __init__(self, spec):
        s = self.spec = spec
        self.mask, self.mask_size = _mask_of(s)
        if s.position is None or s.position.dim != s.rot_dim or s.rot_dim % 2 != 0:
            raise PartError("latent attention turns its whole rotated part: an even rot_dim with a position part as wide")
        self.position = build_part("position", s.position)
        self.q_width = s.heads * (s.head_dim + s.rot_dim)
        self.row = s.rank + s.rot_dim                    # a token's cache row, and a query head after the move
        self.o_width = s.heads * s.value_dim
        self.out_name = "mixer_out"
        # what the choice of a step's entries that make their keys hangs on besides the step (see `_portions`)
        self.rest = f"rest_{self.mask}_{self.mask_size}_{self._made(1)}"
        self.head_gate = getattr(s, "head_gate", None)
        if self.head_gate not in (None, "sigmoid"):
            raise PartError(f"head_gate {self.head_gate!r}: sigmoid or none")
        self.proj = self.o = self.norm = self.uk = self.uk_t = self.uv = self.sink = self.uq = self.q_norm = self.gate = None

    def weight_specs(self):
        s = self.spec
        if s.q_rank is None:
            first = {"q": WeightSpec((self.q_width, s.hidden), stack="down")}
        else:           # the queries' latent comes out of the same projection as the keys' and values'
            first = {"dq": WeightSpec((s.q_rank, s.hidden), stack="down"), "dq.norm": WeightSpec((s.q_rank,), keep_float32=True),
                     "uq": WeightSpec((self.q_width, s.q_rank))}
        specs = {**first, "dkv": WeightSpec((self.row, s.hidden), stack="down"),
                 "dkv.norm": WeightSpec((s.rank,), keep_float32=True),
                 "uk": WeightSpec((s.heads * s.head_dim, s.rank)), "uv": WeightSpec((self.o_width, s.rank)),
                 "o": WeightSpec((s.hidden, self.o_width))}
        if s.sink:
            specs["sink"] = WeightSpec((s.heads,), keep_float32=True, init=("normal", 0.0, 1.0))
        if self.head_gate is not None:      # (with a query latent it rides behind the two latents in the one projection)
            specs["g"] = WeightSpec((s.heads, s.hidden), stack="down" if s.q_rank is not None else None)
        return specs

    def bind(self, weights):
        s = self.spec
        if s.q_rank is None:
            self.proj = stacked([weights["q"], weights["dkv"]])
            self.gate = weights["g"] if self.head_gate is not None else None
        else:
            self.proj = stacked([weights["dq"], weights["dkv"]] + ([weights["g"]] if self.head_gate is not None else []))
            self.uq, self.q_norm = weights["uq"], weights["dq.norm"]
        self.norm = weights["dkv.norm"]
        # the key up-projection as the queries meet it: per head [rank, head_dim]
        self.uk_t = weights["uk"].view(s.heads, s.head_dim, s.rank).transpose(1, 2).contiguous()
        self.uv = weights["uv"].view(s.heads, s.value_dim, s.rank)
        self.uk = weights["uk"]
        self.o = weights["o"]
        self.sink = weights["sink"] if s.sink else None

    def cache_spec(self):
        return PagedSpec((("latent", (1, PAGE, self.row)),), self.mask_size if self.mask is not None else None)

    def libraries(self):
        return ["gemm", "grouped_gemm", "sink_attention", "elementwise"] + _portion_library(self.o)

    def _made(self, keys):
        """Elements that a portion's made rows take: latent and shared parts, keys, values."""
        s = self.spec
        return keys * (self.row + s.heads * s.head_dim + self.o_width)

    def _portions_possible(self, dtype, limits):
        s = self.spec
        return dtype == torch.bfloat16 and s.scale > 0 and (s.head_dim, s.rot_dim, s.value_dim) == (128, 64, 128) and s.rank % 8 == 0 and \
            not limits.get("routed", False)

    def _portions_planned(self, rows, dtype, limits):
        """Elements of `latent_out` for the longest portion that makes its keys (0: none of this runner's does): its place is
        free until the step's other rows come.  Without `limits["spare"]` no more than those other rows need."""
        if not self._portions_possible(dtype, limits) or not limits.get("spare", True):
            return 0
        most = limits["max_length"] if self.mask is None else min(limits["max_length"], self.mask_size + rows)
        return self._made(min(most, PORTION_KEYS) + 64)

    def workspace_plan(self, rows, dtype, limits):
        s = self.spec
        groups = _groups_plan(rows, s.heads, 1, s.rank)
        rest = {(f"{name}_{self.rest}", kind): count for (name, kind), count in groups.items()
                if name.startswith("token_groups") and self._portions_possible(dtype, limits)}
        first = self.q_width if s.q_rank is None else s.q_rank
        more = {} if s.q_rank is None else {("latent_cq", dtype): rows * s.q_rank, ("latent_queries", dtype): rows * self.q_width}
        if self.head_gate is not None:
            more[("latent_gate", dtype)] = rows * s.heads
        return {("latent_proj", dtype): rows * (first + self.row + (s.heads if self.head_gate is not None else 0)),
                ("latent_q", dtype): rows * s.heads * self.row,
                ("latent_out", dtype): max(rows * s.heads * s.rank, self._portions_planned(rows, dtype, limits)), ("attn", dtype): rows * self.o_width,
                (self.out_name, dtype): rows * s.hidden, **more, **rest, **groups}

    def _portions(self, ctx):
        """The step's entries whose keys and values are made for them: (entry, first batch row, tokens, first key, keys).
        For a token the up-projections on the queries' side cost nothing, but then a pair (query, key) is rank + rot + rank
        products a head; with keys and values made once for a portion it is head_dim + rot + value_dim, 1088 against 320 at
        rank 512, for rank * (head_dim + value_dim) products a key and head.  Not in a step that is to be captured: first
        key and number of keys would be fixed in the graph."""
        s = self.spec
        if ctx.routed or ctx.fixed_groups is not None or \
                not ctx.kernels.latent_portions_supported(s.head_dim, s.rot_dim, s.value_dim, s.rank, float(s.scale)):
            return []
        out, room = [], ctx.workspace.room("latent_out", torch.bfloat16)
        for i, (_, row, n, p0) in enumerate(ctx.segments):
            if n < PORTION_ROWS:
                continue
            first = 0 if self.mask is None else max(0, p0 - self.mask_size + 1) if self.mask == "window" else p0 // self.mask_size * self.mask_size
            first = first // 64 * 64                     # (the kernel's blocks of keys start there)
            if PORTION_LEAST_KEYS <= p0 + n - first <= PORTION_KEYS + 64 and self._made(p0 + n - first) <= room:
                out.append((i, row, n, first, p0 + n - first))
        return out

    def _attend_portion(self, ctx, queries, q, pages, view, attn, row, n, first, keys):
        s, k = self.spec, ctx.kernels
        made, at, parts = ctx.workspace.get("latent_out", (self._made(keys),), attn.dtype), 0, []
        for width in (s.rank, s.rot_dim, s.heads * s.head_dim, self.o_width):
            parts.append(made[at:at + keys * width].view(keys, width))
            at += keys * width
        latent, shared, made_k, made_v = parts
        k.latent_rows(pages, view.block_table, ctx.slots, row, first, keys, view.page_size, s.rank, latent, shared)
        # (their number of rows is that of the keys, another one for nearly every portion: on the wide kernel, which needs no
        # plan.  The first prompt of a length, 1000 to 1740 tokens in eight layers of 2048 channels of which two are latent
        # attention: 6.0 ms, with the library's plans for these two products 6.4; one more prompt of that length 3.6 either way)
        k.gemm(latent, self.uk, made_k, library=False)
        k.gemm(latent, self.uv.view(self.o_width, s.rank), made_v, library=False)
        k.portion_attention_split(queries, q, made_k, shared, made_v, ctx.slots, ctx.positions, self.sink, attn, row, n, first,
                                  128 if n * s.heads >= 128 * ctx.compute_units else 64, s.heads, float(s.scale), self.mask, self.mask_size)

    def forward(self, ctx, x, cache_id, write_cache=True):
        s = self.spec
        k = ctx.kernels
        m = x.shape[0]
        ld = self.proj.shape[0]
        proj = ctx.workspace.get("latent_proj", (m, ld), x.dtype)
        k.gemm(x, self.proj, proj)
        view = ctx.cache.paged_view(cache_id)
        pages = view.tensors["latent"]
        q = ctx.workspace.get("latent_q", (m, s.heads * self.row), x.dtype)
        rope, interleaved = _rope_table(self.position, ctx, x.device, s.rot_dim)
        gate = None
        if s.q_rank is None:
            queries, q_ld = proj, ld
            if self.head_gate is not None:
                gate = ctx.workspace.get("latent_gate", (m, s.heads), x.dtype)
                k.gemm(x, self.gate, gate)
            k.latent_prep(proj, q, pages, view.block_table, ctx.slots, ctx.positions, self.norm, float(s.eps), rope, s.heads,
                          s.head_dim, s.rot_dim, s.rank, view.page_size, write_cache, interleaved=interleaved)
        else:
            # the queries' latent: normed in 32-bit over its own root mean square, then up to the heads
            cq = ctx.workspace.get("latent_cq", (m, s.q_rank), x.dtype)
            k.rmsnorm_columns(proj[:, :s.q_rank], self.q_norm, cq, float(s.eps))
            queries, q_ld = ctx.workspace.get("latent_queries", (m, self.q_width), x.dtype), self.q_width
            k.gemm(cq, self.uq, queries)
            if self.head_gate is not None:
                gate = proj[:, s.q_rank + self.row:]
            k.latent_prep(proj[:, s.q_rank:s.q_rank + self.row], q, pages, view.block_table, ctx.slots, ctx.positions, self.norm, float(s.eps),
                          rope, s.heads, s.head_dim, s.rot_dim, s.rank, view.page_size, write_cache, q_src=queries,
                          interleaved=interleaved)
        plain = torch.as_strided(queries, (m, s.heads, s.head_dim), (q_ld, s.head_dim + s.rot_dim, 1), queries.storage_offset())
        attn = ctx.workspace.get("attn", (m, self.o_width), x.dtype)
        portions = self._portions(ctx)
        for _, row, n, first, keys in portions:
            self._attend_portion(ctx, plain, q.view(m, s.heads, self.row)[:, :, s.rank:], pages, view, attn, row, n, first, keys)
        rest = _row_ranges(ctx.segments, tuple(p[0] for p in portions)) if portions else [(0, m)]
        # the others' plain query channels through the key up-projection, head by head, into the first `rank` channels
        moved = torch.as_strided(q, (m, s.heads, s.rank), (s.heads * self.row, self.row, 1), q.storage_offset())
        for r0, r1 in rest:
            k.heads_gemm(plain[r0:r1], self.uk_t, moved[r0:r1])
        if rest:
            lat = ctx.workspace.get("latent_out", (m, s.heads * s.rank), x.dtype)
            attend(ctx, q, pages, pages, view, self.sink, lat, s.heads, 1, self.row, s.rank, float(s.scale), self.mask,
                   self.mask_size, without=tuple(p[0] for p in portions), rest=self.rest)
        for r0, r1 in rest:
            k.heads_gemm(lat.view(m, s.heads, s.rank)[r0:r1], self.uv, attn.view(m, s.heads, s.value_dim)[r0:r1])
        if gate is not None:
            k.head_gate_mul(attn, gate, attn, s.heads)
        out = ctx.workspace.get(self.out_name, (m, s.hidden), x.dtype)
        k.gemm(attn, self.o, out)
        return out
