"""Differential attention of single new tokens that writes their keys and values itself: the same attention and the same pages, to the
bit, as with the writing kernel before it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


# (page; dims that fill their chunks and not; one head set and two; positions at the borders of pages, tiles and ranges; page -1)
@pytest.mark.parametrize("split_keys", [0, 64])
@pytest.mark.parametrize("mask,mask_size", [(None, 0), ("window", 20), ("chunk", 48)])
@pytest.mark.parametrize("heads,kv,dim,vdim,page", [(4, 2, 32, 64, 16), (16, 2, 48, 48, 8), (3, 3, 64, 128, 24)])
def test_a_token_attended_in_the_launch_that_writes_it(heads, kv, dim, vdim, page, mask, mask_size, split_keys):
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16)
    gen = torch.Generator().manual_seed(heads * 100 + page)
    positions = [0, 7, 8, 23, 31, 32, 63, 64, 95, 127, 128, 199]
    n, blocks = len(positions), 200 // page + 1
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()
    # (what a page holds before its key is written must not show: large numbers there; behind the new token too)
    pages = [draw(n * blocks + 1, kv, page, 2 * dim), draw(n * blocks + 1, kv, vdim, page)]
    table = torch.randperm(n * blocks, generator=gen).to(torch.int32).reshape(n, blocks)
    for row, pos in enumerate(positions):
        page_id, at = int(table[row, pos // page]), pos % page
        pages[0][page_id, :, at:] = 3e4
        pages[1][page_id, :, :, at:] = 3e4
    table[4, positions[4] // page] = -1
    table = table.cuda()
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")
    slots, pos = ints(range(n)), ints(positions)
    a, b, c = heads * 2 * dim, kv * 2 * dim, kv * vdim
    proj = draw(n, a + b + c + 8)
    q, keys, values = proj[:, :a], proj[:, a:a + b], proj[:, a + b:a + b + c]
    splits = -(-200 // split_keys) if split_keys else 1
    partial = torch.empty(k.diff_partial_numel(n * 4, heads, vdim, splits), device="cuda")

    def run(in_launch):
        k_pages, v_pages = pages[0].clone(), pages[1].clone()
        out = torch.full((n, heads * vdim), float("nan"), dtype=torch.bfloat16, device="cuda")
        if not in_launch:
            k.diff_kv_write(keys, values, k_pages, v_pages, table, slots, pos, kv, dim, vdim, page)
        k.diff_attention_tiles(q, k_pages, v_pages, table, slots, pos, None, out, partial, slots, torch.ones_like(slots), n, 4, heads,
                               kv, dim, vdim, page, dim ** -0.5, 0.3, 0.8, 1e-5, split_keys=split_keys, max_splits=splits,
                               max_context=200, mask=mask, mask_size=mask_size, own=(keys, values) if in_launch else None)
        return [t.view(torch.int16).cpu().numpy() for t in (out, k_pages, v_pages)], out

    want, _ = run(False)
    got, out = run(True)
    assert torch.isfinite(out).all()
    for x, y in zip(got, want):
        np.testing.assert_array_equal(x, y)
