"""The host-side decisions about attention's key splits, without a GPU: a context whose pages do not fit
one workgroup's page cache is split whatever the batch, and a runner that could not serve its own
max_length is refused when it is built, not in the middle of a step."""
import pytest
import torch

from mini_llm_runtime_amd.config.specs import AttentionSpec, NormSpec, PositionSpec
from mini_llm_runtime_amd.engine.context import StepContext, Workspace
from mini_llm_runtime_amd.kernels.ops import MAX_KEY_SPLITS, MFMA_MAX_PAGES, Kernels
from mini_llm_runtime_amd.parts.registry import PartError, build_part


def kernels_without_gpu(dtype=torch.bfloat16, routed=False):
    k = Kernels.__new__(Kernels)              # the size questions need no device
    k.dtype, k.library_gemm, k.routed, k._libs = dtype, True, routed, {}
    return k


def context(max_context, split_keys=256, split_max_tokens=256):
    ctx = StepContext(kernels_without_gpu(), None, Workspace("cpu"), torch.bfloat16, max_context, split_keys,
                      split_max_tokens)
    ctx.max_context = max_context
    return ctx


@pytest.mark.parametrize("page", [16, 32, 64])
@pytest.mark.parametrize("rows", [1, 64, 300, 4096])
def test_a_context_beyond_the_page_cache_is_split_whatever_the_batch(page, rows):
    longest = Kernels.mfma_longest_context(page)
    assert longest == (MFMA_MAX_PAGES - 2) * page
    ctx = context(longest + 5000)
    keys, splits, partial = ctx.attention_split(rows, rows, 8, 16, 128, longest=longest)
    assert splits > 1 and keys % 64 == 0 and keys <= longest and keys // page + 2 <= MFMA_MAX_PAGES
    assert splits == -(-ctx.max_context // keys) <= MAX_KEY_SPLITS
    assert partial.numel() >= rows * 16 * splits * (128 + 4)
    # at or below the limit a large batch is left alone (it fills the GPU without splits)
    ctx = context(longest)
    assert ctx.attention_split(4096, 4096, 8, 16, 128, longest=longest)[1] == 1


def test_small_batches_over_long_contexts_are_split_and_short_ones_not():
    ctx = context(4096)
    keys, splits, _ = ctx.attention_split(1, 1, 8, 16, 128, longest=65504)
    assert splits > 1 and keys * splits >= 4096
    assert context(200).attention_split(1, 1, 8, 16, 128, longest=65504)[1] == 1
    assert context(4096, split_keys=0).attention_split(1, 1, 8, 16, 128, longest=65504)[1] == 1
    # workgroups enough without a split: none walks more than 2048 keys, and shorter contexts stay whole
    assert context(2048).attention_split(64, 64, 8, 16, 128, longest=65504)[1] == 1
    assert context(2049).attention_split(64, 64, 8, 16, 128, longest=65504)[:2] == (2048, 2)
    assert context(8192).attention_split(64, 64, 8, 16, 128, longest=65504)[:2] == (2048, 4)
    assert context(8192, split_keys=4096).attention_split(64, 64, 8, 16, 128, longest=65504)[:2] == (4096, 2)


class HostUpload:
    """`Uploader` without a GPU."""

    def send(self, values, dst):
        dst[:len(values)] = torch.tensor(values, dtype=torch.int32)


def spelled(hit):
    return [[v[:n].tolist() for v in (first, count)] for first, count, n in hit[:2]] + [hit[2]]


def test_token_groups_that_leave_out_entries_keep_to_themselves():
    """Layers that leave out different entries of one step: what one was handed is not overwritten by the other, and the first
    one's is still there when a third layer leaves out what the first did."""
    ctx = context(4096)
    ctx.workspace.reserve({(f"token_groups_1_{factor}{rest}", torch.int32): 4000 for factor in (0, 4) for rest in ("", "_rest")})
    ctx._group_upload = HostUpload()
    ctx.segments = [(0, 0, 1, 900), (1, 1, 800, 2000), (2, 801, 400, 600), (3, 1201, 150, 0)]
    want = lambda out: [row for i, (_, row, n, _) in enumerate(ctx.segments) if i not in out for row in range(row, row + n)]  # noqa: E731
    covered = lambda hit: sorted(r for first, count, n in hit[:2] for f, c in zip(first[:n].tolist(), count[:n].tolist())  # noqa: E731
                                 for r in range(f, f + c))
    for factor in (0, 4):
        handed = {}
        for out in ((1, 2), (1,), (1, 2), (), (2, 3), (1,)):
            hit = ctx.token_groups(1, factor, out)
            assert covered(hit) == want(out)
            assert handed.setdefault(out, spelled(hit)) == spelled(hit)
        for out in handed:
            assert spelled(ctx.token_groups(1, factor, out)) == handed[out]
    ctx.begin_step()
    ctx.segments = [(0, 0, 40, 0), (1, 40, 3, 5)]
    assert covered(ctx.token_groups(1, 4, (0,))) == [40, 41, 42]


def latent_part(window):
    from mini_llm_runtime_amd.config import config_from_dict
    layer = dict(type="latent_attention", mlp=None, mixer=dict(heads=16, dim=128, rot_dim=64, vdim=128, kv_rank=512, scale=192 ** -0.5,
                                                               rot=dict(dims=64, base=10000.0), mask=dict(size=window)))
    spec = config_from_dict(dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=[layer])).model_spec()
    return build_part("mixer", spec.layers[0].mixer)


def test_latent_layers_of_different_windows_in_one_step():
    """Windows 1024, 256 and 1024 leave other entries of a step to the attention behind the moved queries: every layer's groups
    cover exactly the rows it leaves, out of planned memory, whatever came between."""
    parts = [latent_part(window) for window in (1024, 256, 1024)]
    rows, limits = 1351, dict(max_length=4096, page_size=16, split_keys=256, split_max_tokens=256, target_workgroups=512, max_slots=4)
    ctx = context(4096)
    ctx._group_upload = HostUpload()
    plan = {}
    for part in parts:
        for key, count in part.workspace_plan(rows, torch.bfloat16, limits).items():
            plan[key] = max(plan.get(key, 0), count)
    # (of the large buffers only the room is asked here)
    sizes = {key: count for key, count in plan.items() if key[0].startswith("token_groups")}
    ctx.workspace.reserve(sizes)
    ctx.workspace.room = lambda name, dtype: plan[name, dtype]
    ctx.segments = [(0, 0, 1, 900), (1, 1, 800, 2000), (2, 801, 400, 600), (3, 1201, 150, 0)]
    left = [tuple(p[0] for p in part._portions(ctx)) for part in parts]
    assert left[0] == left[2] != left[1]
    hits = [ctx.token_groups(1, 4, out, part.rest) for part, out in zip(parts, left)]
    for (small, big, _), out in zip(hits, left):
        got = [(f, c) for first, count, n in (small, big) for f, c in zip(first[:n].tolist(), count[:n].tolist())]
        assert sorted(r for f, c in got for r in range(f, f + c)) == \
            [r for i, (_, row, n, _) in enumerate(ctx.segments) if i not in out for r in range(row, row + n)]
    assert ctx.workspace.unplanned_bytes() == 0


@pytest.mark.parametrize("head_dim,value_dim", [(16, 16), (20, 24), (24, 24), (40, 64), (72, 128), (120, 48), (128, 128)])
def test_the_delta_rules_chunks_are_planned_as_the_kernels_lay_them_out(head_dim, value_dim):
    """A step that fills its tokens with one portion, and one of as many portions as there are slots, stay inside the plan."""
    from mini_llm_runtime_amd.config import config_from_dict
    layer = dict(type="channel_delta", mlp=dict(kind="dense", ff=64),
                 mixer=dict(heads=4, kv_heads=2, dim=head_dim, vdim=value_dim, conv=4, decay_rank=16, gate_rank=16))
    spec = config_from_dict(dict(architecture="Tigelorn", vocab=97, width=64, norm=dict(eps=1e-5), layers=[layer],
                                 embedding=dict(bigram=dict(buckets=31, mul_prev=7, mul_cur=29)))).model_spec()
    part, k = build_part("mixer", spec.layers[0].mixer), kernels_without_gpu()
    for rows, slots in ((512, 1), (2048, 1), (2048, 7)):
        plan = part.workspace_plan(rows, torch.bfloat16, dict(max_slots=slots))
        lengths = [rows - 33 * (slots - 1)] + [33] * (slots - 1)
        chunks = sum(-(-n // k.delta_chunk_tokens()) for n in lengths)
        assert plan["delta_chunks", torch.float32] >= k.delta_chunk_floats(chunks, 4, head_dim, value_dim)


def attention_part(head_dim=128):
    norm = NormSpec("rmsnorm", head_dim, 1e-6)
    return build_part("mixer", AttentionSpec("gqa_attention", 1024, 16, 8, head_dim, head_dim ** -0.5, norm,
                                             PositionSpec("rope_split_half", head_dim, 1e6)))


def test_limits_are_checked_when_the_runner_is_built():
    part, k = attention_part(), kernels_without_gpu()
    part.check_limits(k, 40960, 16, 256)                         # the benchmark's sizes
    part.check_limits(k, 65504, 16, 0)                           # fits without splits
    with pytest.raises(PartError, match="needs key splits"):
        part.check_limits(k, 65505, 16, 0)
    with pytest.raises(PartError, match="exceeds"):
        part.check_limits(k, 1 << 20, 16, 1 << 17)
    part.check_limits(k, 1 << 20, 16, 256)
    with pytest.raises(PartError, match="more than"):
        part.check_limits(k, (1 << 15) * MAX_KEY_SPLITS + 1, 16, 256)
    # the float engine's kernel walks the block table itself
    part.check_limits(kernels_without_gpu(torch.float32), 1 << 22, 16, 0)


def test_even_head_sizes_are_taken_and_odd_ones_refused():
    for d in (2, 6, 20, 34, 256):
        attention_part(d)
    for d in (15, 258):
        with pytest.raises(PartError, match="head_dim"):
            attention_part(d)


def test_the_planned_partial_results_hold_every_choice_of_splits():
    """The 8B sizes with requests of up to 40960 tokens: whatever the step (single tokens, a 2048-token portion
    behind 34816 tokens of context, one single token beside such a portion), the partial results of split
    attention stay within what the part planned for them, and a forced split still covers the context."""
    spec = AttentionSpec("gqa_attention", 4096, 32, 8, 128, 128 ** -0.5, NormSpec("rmsnorm", 128, 1e-6),
                         PositionSpec("rope_split_half", 128, 1e6))
    part = build_part("mixer", spec)
    rows, page = 2048 + 64, 16
    limits = dict(max_length=40960, page_size=page, split_keys=256, split_max_tokens=256, target_workgroups=512)
    planned = part.workspace_plan(rows, torch.bfloat16, limits)[("attn_partial", torch.float32)]
    tiles_longest, mfma_longest = Kernels.tiles_longest_context(page), Kernels.mfma_longest_context(page)
    assert limits["max_length"] > tiles_longest          # prompt portions are split for every row at this length
    seen = 0
    for context in (300, 4096, 20000, tiles_longest, tiles_longest + 1, 34816 + 2048, 40960):
        ctx = context_with_budget(context, planned)
        for units_rows, batch_rows in ((1, 1), (8, 8), (64, 64), (1, rows), (8, rows), (200, rows)):
            keys, splits, partial = ctx.attention_split(units_rows, batch_rows, 8, 32, 128, longest=mfma_longest)
            assert partial is None or partial.numel() <= planned
            assert splits == 1 or keys * splits >= context
            seen = max(seen, 0 if partial is None else partial.numel())
        for groups in (1, 16, 128):                        # groups of a prompt portion (16 tokens x 4 heads a kv head)
            keys, splits, partial = ctx.group_split(groups, rows, 8, 32, 128, longest=tiles_longest)
            assert partial is None or partial.numel() <= planned
            if context > tiles_longest:
                assert splits > 1 and keys <= tiles_longest and keys * splits >= context
            seen = max(seen, 0 if partial is None else partial.numel())
    assert seen == planned                                 # the plan is met by some step, not merely an upper bound
    assert ctx.workspace.unplanned_bytes() <= 4 * planned  # (this workspace has no plan: one buffer, never beyond it)


def context_with_budget(max_context, budget):
    ctx = context(max_context)
    ctx.partial_budget = budget
    return ctx


def test_a_smallest_key_range_beyond_the_portion_kernels_reach_is_refused_when_the_runner_is_built():
    part, k = attention_part(), kernels_without_gpu()
    longest = Kernels.tiles_longest_context(16)
    part.check_limits(k, 40960, 16, longest - longest % 64)
    with pytest.raises(PartError, match="prompt portions"):
        part.check_limits(k, 40960, 16, 49152)             # fits the single-token kernel, not the portions'
    with pytest.raises(PartError, match="prompt portions"):
        part.check_limits(k, 4096, 16, 49152)              # refused whatever max_length: splits also fill the GPU
    # pages that the portion kernel does not take (no power of two) leave only the other kernel's limit
    part.check_limits(k, 40960, 48, 49152)


def test_key_ranges_of_one_width_whatever_the_batch():
    """The float engine's attention (`StepContext.fixed_split`): the width of a key range is the runner's setting
    for every number of rows and every context (so a token's sums do not depend on the batch), the ranges cover
    the context, and rows whose partial results would not fit what was planned are served by several launches."""
    per = lambda splits: Kernels.attention_partial_numel(1, 16, 128, splits)
    for max_context in (100, 256, 257, 4096, 40960):
        for rows in (1, 7, 300, 2048):
            ctx = context_with_budget(max_context, 2 * 512 * 128 * 132)
            keys, splits, chunk, partial = ctx.fixed_split(rows, 16, 128)
            if max_context <= 256:
                assert (keys, splits, chunk, partial) == (0, 1, rows, None)
                continue
            assert keys == 256 and splits == -(-max_context // 256)
            assert 1 <= chunk <= rows and partial.numel() == chunk * per(splits) <= ctx.partial_budget
            assert chunk == rows or (chunk + 1) * per(splits) > ctx.partial_budget
    # beyond 1024 ranges the width doubles (the merge kernel keeps one weight a range in LDS)
    ctx = context_with_budget(300000, None)
    keys, splits, chunk, _ = ctx.fixed_split(3, 16, 128)
    assert keys == 512 and splits == -(-300000 // 512) <= MAX_KEY_SPLITS and chunk == 3


@pytest.mark.parametrize("rows,max_context,keys,wide,of_64,of_320", [
    (1, 512, 64, 256, 64, 320), (1, 257, 64, 256, 64, 0), (1, 1280, 64, 256, 64, 320), (1, 1281, 128, 256, 64, 320), (1, 2560, 128, 256, 64, 320),
    (1, 2561, 256, 256, 64, 320), (6, 512, 64, 256, 64, 320), (7, 512, 128, 256, 64, 320), (12, 512, 128, 256, 64, 320), (13, 512, 256, 256, 64, 320),
    (3, 2048, 128, 256, 64, 320), (4, 2048, 256, 256, 128, 320), (8, 4096, 512, 512, 512, 320), (1, 256, 0, 0, 64, 0)])
def test_few_workgroups_take_narrower_key_ranges(rows, max_context, keys, wide, of_64, of_320):
    """Half the setting's width (256) while that is no more than three workgroups to two compute units and twenty ranges.  A model that
    routes (`wide`), a setting whose half is no multiple of 64 (320) and one that is narrow already (64) are never narrowed: their ranges
    are the setting's, or wider ones where those still fill the GPU.  (0: one workgroup walks every key.)"""
    def split(base, routed=False):
        ctx = context(max_context, split_keys=base)
        ctx.compute_units, ctx.routed = 256, routed
        return ctx.attention_split(rows, rows, 8, 16, 128, longest=65504)[:2]
    ranges = lambda width: (width, -(-max_context // width) if width else 1)  # noqa: E731
    assert split(256) == ranges(keys) and split(256, routed=True) == ranges(wide)
    assert split(64) == split(64, routed=True) == ranges(of_64)
    assert split(320) == split(320, routed=True) == ranges(of_320)


@pytest.mark.parametrize("lengths,keys", [([1], 64), ([2], 64), ([1, 1], 64), ([3], 256), ([2, 1], 256), ([5], 256), ([1] * 6, 256), ([400, 2], 64), ([400, 3], 256)])
def test_short_portions_keep_the_settings_key_ranges(lengths, keys):
    """What single tokens alone gain by (they have a kernel of their own) costs portions of several tokens."""
    part, ctx = attention_part(), context(512)
    ctx.workspace.reserve({("token_groups_8_4", torch.int32): 4000})
    ctx._group_upload, ctx.n_tokens, ctx.routed, ctx.compute_units = HostUpload(), sum(lengths), False, 256
    ctx.segments = [(i, sum(lengths[:i]), n, 0) for i, n in enumerate(lengths)]
    ctx.slots = ctx.positions = torch.zeros(sum(lengths), dtype=torch.int32)
    taken = []
    ctx.kernels.profiler = None
    ctx.kernels.attention_mfma = lambda *a, **kw: taken.append((kw["split_keys"], kw["max_splits"]))
    ctx.kernels.attention_tiles = lambda *a, **kw: None
    part._work = None
    pages = torch.empty((70, 8, 16, 128), dtype=torch.bfloat16)
    view = type("View", (), dict(k_pages=pages, v_pages=pages, block_table=None, page_size=16))
    part._attend_cached(ctx, torch.empty((sum(lengths), 16 * 128), dtype=torch.bfloat16), view)
    assert taken == [(keys, 512 // keys)]


@pytest.mark.parametrize("units,max_context,short,routed,keys", [
    (32, 2048, True, False, 128), (32, 2724, True, False, 256), (16, 2724, True, False, 128), (4, 2048, True, False, 64), (4, 4096, True, False, 128),
    (4, 4097, True, False, 256), (32, 2048, False, False, 256), (32, 2048, True, True, 256), (64, 512, True, False, 64), (128, 512, True, False, 128),
    (512, 2048, True, False, 0), (4, 256, True, False, 0)])
def test_differential_attention_of_few_short_groups_takes_narrower_key_ranges(units, max_context, short, routed, keys):
    from mini_llm_runtime_amd.parts.diff_attention import DiffAttention
    part = object.__new__(DiffAttention)
    part.spec, part.mask, part._page_size = type("Spec", (), dict(q_heads=16, value_dim=128)), None, 16
    ctx = context(max_context)
    ctx.routed = routed
    found = part._tile_splits(ctx, units, 4 * units, 1 << 40, short)
    assert found == ((keys, -(-max_context // keys)) if keys else (0, 1))


@pytest.mark.parametrize("sizes", [(17, 6144, 2048), (64, 12288, 1024), (333, 768, 2048), (1777, 4096, 18432), (1603, 28736, 6016), (653, 23648, 2176)])
def test_products_of_a_model_with_a_router_keep_the_order_of_their_sums(sizes):
    """Where the vendor library may add in another order than the many-row kernel, a model that chooses among experts stays with
    it (asked without a GPU: the answer must not need the kernels' library); other models ask the kernels' own rule."""
    k = kernels_without_gpu()
    k._wide_choices = {sizes + (None,): True, sizes + ("silu",): True}
    assert k.wide_product(*sizes) and k.wide_product(*sizes, "silu")
    k = kernels_without_gpu(routed=True)
    k._wide_choices = {sizes + (None,): True, sizes + ("silu",): True}
    assert not k.wide_product(*sizes) and not k.wide_product(*sizes, "silu")
    k._wide_choices.update({(1777, 4096, 4096, None): True, (1777, 6144, 4096, None): True, (1777, 3000, 2048, "silu"): True, (1777, 6000, 2048, "silu"): True})
    assert k.wide_product(1777, 4096, 4096) and not k.wide_product(1777, 6144, 4096)
    assert k.wide_product(1777, 3000, 2048, "silu") and not k.wide_product(1777, 6000, 2048, "silu")     # (a gate's outputs are two)


@pytest.mark.parametrize("mask,size", [("window", 512), ("chunk", 1), ("window", 100000), (None, 0)])
@pytest.mark.parametrize("units", [1, 4, 16, 32, 200])
def test_narrower_key_ranges_of_differential_attention_are_few_behind_a_mask_too(units, mask, size):
    """Ranges are launched for the whole context, whatever part of it a mask lets a workgroup walk: what narrowing adds stays within its
    32 ranges and its number of workgroups, and a long context behind a short window has the ranges of the setting."""
    from mini_llm_runtime_amd.parts.diff_attention import DiffAttention
    part = object.__new__(DiffAttention)
    part.spec, part.mask, part.mask_size, part._page_size = type("Spec", (), dict(q_heads=16, value_dim=128)), mask, size, 16
    for max_context in (200, 600, 1100, 2048, 4096, 4097, 8192, 8193, 32768):
        ctx = context(max_context)
        ctx.routed = False
        keys, splits = part._tile_splits(ctx, units, 4 * units, 1 << 40, True)
        if splits == 1:
            continue
        wide = part._tile_splits(ctx, units, 4 * units, 1 << 40, False)
        assert splits == -(-max_context // keys)
        assert (keys, splits) == wide or (keys < 256 and splits <= 32 and units * splits <= ctx.target_workgroups)


@pytest.mark.parametrize("m,n,kk,act,taken,one_sum,few", [
    (33, 5632, 2112, None, True, True, False), (64, 8192, 4096, "silu", True, True, False), (32, 8448, 2112, None, True, True, False),
    (33, 5624, 2112, None, False, True, False), (32, 8192, 2112, None, False, True, False), (64, 16448, 4096, None, False, True, False),
    (64, 5632, 4160, None, False, True, False), (33, 2816, 2112, "silu", True, True, False), (33, 5632, 2112, "gelu_erf", True, True, False),
    (32, 8448, 2048, None, False, False, True), (64, 8448, 1024, "silu", False, False, True), (16, 8448, 2048, None, False, False, False)])
def test_up_to_64_rows_of_a_model_with_a_router(m, n, kk, act, taken, one_sum, few):
    """In place of the library tiles of one sum over k, where it adds so; in place of the kernels that stream the weight the narrow
    tiles, whose sums are theirs.  (Asked with the kernels' own rule always answering yes.)"""
    k = kernels_without_gpu(routed=True)
    k._wide_choices = {(m, n, kk, act): True, (m, n, kk, act, "few"): True}
    assert (k.wide_product(m, n, kk, act), k.one_sum(m, kk), k.few_product(m, n, kk, act)) == (taken, one_sum, few)


@pytest.mark.parametrize("shift_q,shift_out", [(0, 0), (1, 0), (0, 1)])
def test_rows_that_do_not_start_on_16_bytes_keep_the_attention_that_takes_them(shift_q, shift_out):
    """Queries or results that are views off 16 bytes: the prompt portions' kernel for whole rows does not take them, the general one
    does, and nothing is refused."""
    from mini_llm_runtime_amd.parts.sink_attention import attend
    ctx = context(1000)
    ctx.workspace.reserve({("token_groups_1_8", torch.int32): 4000})
    ctx._group_upload, ctx.segments, ctx.n_tokens, ctx.routed = HostUpload(), [(0, 0, 300, 0)], 300, True
    ctx.slots = ctx.positions = torch.zeros(300, dtype=torch.int32)
    ctx.max_positions, ctx.compute_units = 1000, 256
    taken = []
    k = ctx.kernels
    k.sink_attention_rows = lambda *a, **kw: taken.append("rows")
    k.sink_attention_tiles = lambda *a, **kw: taken.append("tiles")

    def rows(width, shift):
        return torch.empty(300 * width + shift, dtype=torch.bfloat16)[shift:].view(300, width)
    k_pages, v_pages = (torch.empty((70, 1, 16, 128), dtype=torch.bfloat16) for _ in range(2))
    view = type("View", (), dict(page_size=16, block_table=None))
    attend(ctx, rows(16 * 128, shift_q), k_pages, v_pages, view, None, rows(16 * 128, shift_out), 16, 1, 128, 128, 0.1, None, 0)
    assert taken[0] == ("tiles" if shift_q or shift_out else "rows")


def test_whether_a_model_routes_is_said_where_its_kernels_are_made(monkeypatch):
    """No state of the class, and none that is set from outside later."""
    monkeypatch.setattr(torch.cuda, "is_available", lambda: True)
    assert not hasattr(Kernels, "routed")
    assert Kernels(torch.bfloat16, routed=True).routed and not Kernels(torch.bfloat16).routed


@pytest.mark.parametrize("library", [True, False])
def test_heads_in_the_products_epilogue_only_where_their_tile_is_worth_it(library):
    """Narrow products leave most of the chip idle in tiles of whole heads: they keep the best tile and the launch behind it, whether the
    vendor library stands beside the kernel or not."""
    k = kernels_without_gpu()
    k.library_gemm, k._wide_choices = library, {}
    assert all(k.qkv_product(m, q, kv, 128, inner, 16) for m, q, kv, inner in ((2048, 16, 8, 1024), (1024, 16, 8, 1024), (333, 32, 8, 4096)))
    assert not any(k.qkv_product(m, q, kv, 128, inner, 16) for m, q, kv, inner in ((83, 7, 1, 5120), (256, 32, 8, 4096), (99, 16, 2, 5120), (128, 24, 8, 2560)))


@pytest.mark.parametrize("rows,n,k,experts,shape", [
    (160, 4096, 448, 8, 4), (160, 4096, 384, 8, -1), (161, 4096, 448, 8, 5), (447, 4096, 384, 8, -1), (320, 2048, 448, 16, 4), (320, 2112, 448, 16, -1),
    (320, 2112, 640, 16, -1), (320, 2112, 704, 16, 4), (640, 4096, 640, 32, -1), (640, 4096, 64, 33, 4), (8, 128, 64, 256, 4), (448, 2048, 64, 8, 5),
    (1023, 2048, 64, 8, 5), (447, 2048, 64, 8, -1), (448, 2112, 64, 8, -1), (448, 128, 64, 2, 0), (64, 100, 1024, 2, -1), (64, 128, 1000, 2, -1)])
def test_products_of_experts_with_few_rows(rows, n, k, experts, shape):
    """Both sides of every line: a short k of up to 32 experts, the rows a tile holds, tiles that are no more than compute units."""
    from mini_llm_runtime_amd.kernels import build
    assert build.load("grouped_gemm", torch.bfloat16).mlr_experts_shape(rows, n, k, experts) == shape
