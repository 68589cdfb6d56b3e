"""The page of a key without a division (csrc/pages.h): for every page size, on the CPU; and attention over pages of a size that is no
power of two at contexts where the high word of one product would name the page behind."""
import pytest
import torch


@pytest.mark.parametrize("size", [1, 2, 7, 8, 24, 48, 1000, 65535, 65536, 65537, 100000, 163840, (1 << 20) + 8, (1 << 30) - 1, 1 << 30, (1 << 31) - 1])
def test_every_key_is_found_in_its_page(size):
    """Both sides of the edges between pages, the first ones and the last below 2^31."""
    from mini_llm_runtime_amd.kernels import build
    page_of = build.load("diff_attention", torch.bfloat16).mlr_page_of_key
    last = (1 << 31) - 1
    edges = {q * size for n in (1, 3, 1000, last // size // 2, last // size) for q in (n - 1, n, n + 1)}
    for key in sorted({min(max(e + d, 0), last) for e in edges | {last} for d in (-2, -1, 0, 1)}):
        assert page_of(size, key) == key // size, key


@pytest.mark.gpu
def test_the_last_keys_of_a_long_page_that_is_no_power_of_two():
    """One page of 163840 tokens, and two of 100000: the bits of pages of 2^13 (the same tiles of keys).  A
    window of 40 keys, so that each of them counts."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16)
    ints = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    for size, total in ((163840, 163840), (100000, 200000)):
        n, window, dim = 3, 40, 16
        blocks = -(-total // 8192)
        gen = torch.Generator("cuda").manual_seed(size)
        rnd = lambda *shape: torch.randn(*shape, generator=gen, device="cuda").to(torch.bfloat16)  # noqa: E731
        keys, values, q = rnd(blocks * 8192, 2 * dim), rnd(blocks * 8192, dim), rnd(n, 4 * dim)
        slots, pos = ints(0, 0, 0), ints(*range(total - n, total))
        got = []
        for page in (8192, size):
            pages = -(-total // page)
            room = max(pages * page, blocks * 8192)
            wide = lambda t: torch.cat([t, torch.zeros(room - t.shape[0], t.shape[1], dtype=t.dtype, device="cuda")])[:pages * page]  # noqa: E731
            table = ints(*range(pages), -1)[None].contiguous()
            kp, vp = wide(keys).view(pages, 1, page, 2 * dim), wide(values).view(pages, 1, page, dim)
            outs = []
            for ranges in (0, 4096):
                splits = -(-total // ranges) if ranges else 1
                out = torch.full((n, 2 * dim), float("nan"), dtype=torch.bfloat16, device="cuda")
                partial = torch.full((k.diff_partial_numel(4, 2, dim, splits),), float("nan"), device="cuda")
                k.diff_attention_tiles(q, kp, vp.transpose(2, 3).contiguous(), table, slots, pos, None, out, partial, ints(0), ints(n), 1, 4, 2, 1, dim,
                                       dim, page, 0.3, 0.5, 0.8, 1e-5, split_keys=ranges, max_splits=splits, max_context=total, mask="window",
                                       mask_size=window)
                outs.append(out)
            out = torch.full((n, 2 * dim), float("nan"), dtype=torch.bfloat16, device="cuda")
            k.sink_attention_tiles(q, kp, vp, table, slots, pos, None, out, ints(0), ints(n), 1, 2, True, 2, 1, 2 * dim, dim, page, 0.3, "window", window,
                                   total)
            got.append([*outs, out])
        for small, large in zip(*got):
            assert torch.isfinite(small.float()).all() and torch.equal(small.view(torch.int16), large.view(torch.int16)), size
