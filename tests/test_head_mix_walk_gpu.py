"""Attention whose heads are mixed, in one walk over the keys (`Kernels.head_mix_walk`), against the formula in 64 bits."""
import numpy as np
import pytest
import torch

from test_nuvorax_gpu import back, ints, paged, plain_attend, rounded, tolerance, turn_table

pytestmark = pytest.mark.gpu


def launch(k, q, k_pages, v_pages, table, slots, pos, talk, sink, v_rope, gate, heads, kv, dim, page, scale, cap, first, count, tokens,
           context, keys):
    """NaN in every piece of scratch memory and in the output."""
    ranges, n = -(-context // keys), len(first)
    rows = n * ranges * k.head_mix_walk_rows(kv, tokens)
    nan = lambda size: torch.full((size,), float("nan"), device="cuda")  # noqa: E731
    out = torch.full((q.shape[0], heads * 128), float("nan"), dtype=q.dtype, device="cuda")
    part = (ints(first), ints(count), n, keys, ranges, nan(rows) if ranges > 1 else None, nan(rows * kv * 128) if ranges > 1 else None)
    k.head_mix_walk(q, k_pages, v_pages, table, slots, pos, talk, sink, v_rope, gate, out, part if tokens == 4 else None,
                    part if tokens == 1 else None, heads, kv, dim, 128, page, scale, cap)
    return back(out)


@pytest.mark.parametrize("sink", [None, -1.5, "learned"])
@pytest.mark.parametrize("kv,dim,page", [(4, 128, 16), (4, 128, 64), (2, 128, 8), (2, 128, 32), (1, 128, 16), (1, 128, 256)])
def test_every_position_in_groups_and_ranges(sink, kv, dim, page):
    """A request of 267 tokens (over the edges of blocks of 64 and 128 keys and of ranges, the last of 11 keys), in groups of four, of
    three, with a ragged last one, and of single tokens, its keys whole and in ranges; with and without turned values, in both pairings,
    and gates.  Tolerance: that of the other matrix-core form, whose weights are rounded to bfloat16 three times for this one's once."""
    from mini_llm_runtime_amd.kernels import Kernels
    rng = np.random.default_rng(12)
    T, cap, heads = 267, 12.0, 4 * kv
    scale = 0.7 * (dim / 128) ** -0.5
    k = Kernels(torch.bfloat16)
    bf = lambda *shape: rounded(rng.normal(size=shape), torch.bfloat16)  # noqa: E731
    keys, values, q, gate = bf(T, kv, dim), bf(T, kv, 128), bf(T, heads, dim), bf(T, heads)
    talk = rounded(rng.normal(size=(heads, heads)) * heads ** -0.5, torch.float32)
    sinks = rounded(rng.normal(size=heads), torch.float32) if sink == "learned" else sink
    k_pages, v_pages, table = paged(back(keys), back(values), page, torch.bfloat16, seed=3)
    slots, pos = torch.zeros(T, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")
    for turned, gated in ((True, True), (False, False)):
        want = plain_attend(back(q), back(keys), back(values), np.arange(T), scale, cap, back(sinks) if sink == "learned" else sink,
                            back(talk), 50.0 if turned else None, back(gate) if gated else None)
        v_rope = (turn_table(128, 50.0, T), False) if turned else None
        for tokens, size, span in ((4, 4, 384), (4, 3, 384), (4, 4, 128), (1, 1, 384), (1, 1, 128)):
            first = list(range(0, T, size))
            got = launch(k, q.view(T, -1), k_pages, v_pages, table, slots, pos, talk, sinks, v_rope, gate if gated else None, heads, kv, dim,
                         page, scale, cap, first, [min(size, T - f) for f in first], tokens, T, span)
            np.testing.assert_allclose(got, want, err_msg=str((turned, tokens, size, span)), **tolerance("bfloat16"))


def test_values_in_neighbouring_pairs_and_scores_at_the_cap():
    """Value channels turned in pairs (2 j, 2 j + 1), and one key at the cap of 60 among keys far below it."""
    from mini_llm_runtime_amd.config.specs import PositionSpec
    from mini_llm_runtime_amd.kernels import Kernels
    from mini_llm_runtime_amd.parts.rope import Rope
    rng = np.random.default_rng(4)
    T, kv, dim, page, heads = 150, 4, 128, 16, 16
    k = Kernels(torch.bfloat16)
    keys, values = rounded(rng.normal(size=(T, kv, dim)), torch.bfloat16), rounded(rng.normal(size=(T, kv, 128)), torch.bfloat16)
    q = np.zeros((T, heads, dim))
    for i in range(T):
        q[i] = np.repeat(back(keys)[(7 * i) % (i + 1)], 4, axis=0) * 4.0
    q = rounded(q, torch.bfloat16)
    talk = rounded(rng.normal(size=(heads, heads)) * 0.25, torch.float32)
    k_pages, v_pages, table = paged(back(keys), back(values), page, torch.bfloat16)
    slots, pos = torch.zeros(T, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")
    v_rope = (Rope(PositionSpec("rope", 128, 9.0, interleaved=True)).rotation(T, "cuda").table, True)
    halves = plain_attend(back(q), back(keys), back(values), np.arange(T), 1.0, 60.0, 0.0, back(talk), None, None).reshape(T, heads, 128)
    import plain.nuvorax_plain as P
    turned = P.rotate_values(np.concatenate([halves[..., 0::2], halves[..., 1::2]], axis=-1), np.arange(T), 9.0, -1.0)
    want = np.stack([turned[..., :64], turned[..., 64:]], axis=-1).reshape(T, -1)
    for tokens, size, span in ((4, 4, 256), (1, 1, 128)):
        first = list(range(0, T, size))
        got = launch(k, q.view(T, -1), k_pages, v_pages, table, slots, pos, talk, 0.0, v_rope, None, heads, kv, dim, page, 1.0, 60.0, first,
                     [min(size, T - f) for f in first], tokens, T, span)
        np.testing.assert_allclose(got, want, **tolerance("bfloat16"))


@pytest.mark.parametrize("kv", [4, 2, 1])
def test_groups_and_single_tokens_of_one_launch(kv):
    """The bits of a launch of their own, whichever of the two has its keys in ranges."""
    from mini_llm_runtime_amd.kernels import Kernels
    rng = np.random.default_rng(2)
    T, page, heads = 300, 16, 4 * kv
    k = Kernels(torch.bfloat16)
    keys, values, q = (rounded(rng.normal(size=(T, n, 128)), torch.bfloat16) for n in (kv, kv, heads))
    talk = rounded(rng.normal(size=(heads, heads)) * 0.25, torch.float32)
    k_pages, v_pages, table = paged(back(keys), back(values), page, torch.bfloat16)
    slots, pos = torch.zeros(T, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")
    split = 130
    first4, first1 = list(range(split, T, 4)), list(range(split))
    count4 = [min(4, T - f) for f in first4]
    for keys4, keys1 in ((384, 384), (128, 384), (384, 128), (128, 256)):
        args = (k, q.view(T, -1), k_pages, v_pages, table, slots, pos, talk, None, None, None, heads, kv, 128, page, 0.09, 30.0)
        want = np.concatenate([launch(*args, first1, [1] * split, 1, T, keys1)[:split], launch(*args, first4, count4, 4, T, keys4)[split:]])
        parts = []
        for first, count, tokens, span in ((first4, count4, 4, keys4), (first1, [1] * split, 1, keys1)):
            ranges = -(-T // span)
            rows = len(first) * ranges * k.head_mix_walk_rows(kv, tokens)
            parts.append((ints(first), ints(count), len(first), span, ranges, torch.full((rows,), float("nan"), device="cuda"),
                          torch.full((rows * kv * 128,), float("nan"), device="cuda")))
        out = torch.full((T, heads * 128), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.head_mix_walk(q.view(T, -1), k_pages, v_pages, table, slots, pos, talk, None, None, None, out, *parts, heads, kv, 128, 128, page,
                        0.09, 30.0)
        assert np.array_equal(back(out), want)


def test_the_launch_shapes_fit_their_scratch_memory():
    """Ranges and groups a launch for every kind of step stay within the planned buffers, hold the context and come in whole blocks."""
    from mini_llm_runtime_amd.parts.head_mix_attention import GROUP, MOST_RANGES, PARTIAL_CAP, SUMS_CAP, walk_shape
    for kv in (1, 2, 4):
        for tokens in (1, 4):
            for groups in (1, 2, 3, 64, 175, 600, 5000):
                for context in (1, 64, 129, 700, 2500, 16385, 262144):
                    keys, ranges, some, rows = walk_shape(kv, groups, tokens, context, 256)
                    assert keys % 128 == 0 and keys * ranges >= context > keys * (ranges - 1) and 1 <= some <= groups and ranges <= MOST_RANGES
                    if ranges > 1:
                        batch = groups * (2 if tokens == 4 else 1)          # the fewest rows that make so many groups
                        assert some * ranges * rows * kv * 128 <= min(PARTIAL_CAP, batch * GROUP * 4 * kv * 128 * MOST_RANGES)
                        assert some * ranges * rows <= min(SUMS_CAP, batch * GROUP * 16 * MOST_RANGES)
