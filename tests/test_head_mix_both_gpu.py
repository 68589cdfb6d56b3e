"""Attention whose heads are mixed, groups of a prompt portion and single tokens in the launches of one of them: the bits of launches of
their own."""
import numpy as np
import pytest
import torch

from test_nuvorax_gpu import back, ints, paged, rounded, turn_table

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,kv,dim,vdim,page", [(16, 4, 128, 128, 16), (32, 8, 64, 128, 8), (9, 3, 40, 48, 24), (4, 1, 64, 16, 16), (12, 4, 128, 256, 16)])
def test_bits_of_launches_of_their_own(heads, kv, dim, vdim, page):
    """A ragged last group, ranges that end inside a tile of keys, every number of kv heads a workgroup, either with its keys in ranges
    of their own; three heads a kv head leave places empty."""
    from mini_llm_runtime_amd.kernels import Kernels
    rng = np.random.default_rng(5)
    T, split, cap = 333, 150, 20.0
    k = Kernels(torch.bfloat16)
    assert k.head_mix_both_supported(heads, kv, dim, vdim, page, cap)
    keys, values, q = (rounded(rng.normal(size=(T, n, d)), torch.bfloat16) for n, d in ((kv, dim), (kv, vdim), (heads, dim)))
    talk, gate = rounded(rng.normal(size=(heads, heads)) * 0.3, torch.float32), rounded(rng.normal(size=(T, heads)), torch.bfloat16)
    k_pages, v_pages, table = paged(back(keys), back(values), page, torch.bfloat16)
    slots, pos = torch.zeros(T, dtype=torch.int32, device="cuda"), torch.arange(T, dtype=torch.int32, device="cuda")
    v_rope = (turn_table(vdim, 50.0, T), False)
    pad, inner, most = k.head_mix_layout(heads, kv, vdim)
    first16, first1 = list(range(split, T, 16)), list(range(split))
    groups = ((first16, [min(16, T - f) for f in first16], 16), (first1, [1] * split, 1))
    ktiles = -(-T // 32)
    before = (q.view(T, -1), k_pages, v_pages, table, slots, pos, talk, 0.0, v_rope, gate)
    sizes = (heads, kv, dim, vdim, page, 0.3, cap)
    nan = lambda n, dtype=torch.float32: torch.full((n,), float("nan"), dtype=dtype, device="cuda")  # noqa: E731
    for score_keys, value_keys, one_score, one_value, block, one_block in ((352, 352, 352, 512, 8, 1), (128, 96, 256, 256, 1, 8), (64, 352, 128, 512, 2, 2)):
        launches = []
        for (first, count, tokens), sk, vk, b in zip(groups, (score_keys, one_score), (value_keys, one_value), (block, one_block)):
            rows, sr, vr = len(first) * tokens, -(-ktiles * 32 // sk), -(-ktiles * 32 // vk)
            launches.append((ints(first), ints(count), len(first), nan(rows * ktiles * 32 * inner, torch.bfloat16), nan(rows * inner * sr),
                             nan(rows * heads * vr * vdim), ktiles, sk, sr, vk, vr, min(b, most)))
        want, got = (torch.full((T, heads * vdim), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
        for (first, count, n, *rest), (_, _, tokens) in zip(launches, groups):
            k.head_mix_tiles(*before, want, first, count, n, tokens, *sizes, *rest)
        for launch in launches:
            for scratch in launch[3:6]:
                scratch.fill_(float("nan"))
        k.head_mix_tiles_both(*before, got, *launches, *sizes)
        assert torch.isfinite(want.float()).all() and torch.equal(got.view(torch.int16), want.view(torch.int16))
