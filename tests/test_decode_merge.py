"""Decoding attention whose last workgroup merges the key ranges: even ranges (the host's rule is the kernel's, they cover every
context), and the kernel against the plain attention at the edges of ranges, tiles and groups of heads."""
import ctypes
import math

import pytest
import torch

from mini_llm_runtime_amd.engine.context import StepContext, Workspace
from mini_llm_runtime_amd.kernels import build
from mini_llm_runtime_amd.kernels.ops import KernelError


def test_the_hosts_rule_of_even_ranges_is_the_kernels_and_never_falls():
    lib = build.load("attention", torch.bfloat16)
    for units in (1, 3, 8, 24, 40, 64, 96, 128):
        wide = -(-2048 * 256 // units // 64) * 64
        last = 0
        for walk in [*range(1, 400, 7), 511, 512, 513, 1024, 2047, 2048, 2049, 4096, 4931, 5461, 5462, 8192, 40960, 131072, 700000]:
            n = StepContext.even_ranges(walk, 256, units, wide)
            assert n == lib.mlr_attention_even_ranges(*(ctypes.c_int(v) for v in (walk, 256, units, wide)))
            width = -(-(-(-walk // 64)) // n) * 64
            assert last <= n <= -(-walk // 64) and n * width >= walk
            assert width <= 2 * wide * units // 256 + 128          # what the kernel's launch checks against a workgroup's page ids
            last = n


def test_counters_are_zeros_when_they_are_made_and_when_they_grow():
    ws = Workspace("cpu")
    ws.reserve({("hidden", torch.float32): 100, ("arrivals", torch.int32): 24})
    assert ws.get("arrivals", (24,), torch.int32).eq(0).all() and ws.unplanned_bytes() == 0
    assert ws.get("arrivals", (9000,), torch.int32).eq(0).all()


def fused_entry(groups, kv_heads, head_dim, page, split_keys, max_splits, workgroups, max_context):
    """The kernel's entry with sizes only: for calls that it refuses, which look at no address."""
    lib, some = build.load("attention", torch.bfloat16), ctypes.c_void_p(256)
    ints = lambda *values: [ctypes.c_int(v) for v in values]
    return lib.mlr_attention_decode_fused(some, *ints(3 * kv_heads * head_dim), some, some, some, *ints(1 << 20), some, some, some, some, some, some,
                                          *ints(groups, kv_heads, kv_heads, head_dim, page, 0), ctypes.c_float(1.0),
                                          *ints(split_keys, max_splits, workgroups, max_context), None, None, ctypes.c_float(0.0), None, some, None)


@pytest.mark.parametrize("max_splits,page,max_context", [(1, 32, 4094 * 32 + 1), (1, 64, 300000), (2, 48, 2 * 4096 * 48 - 64), (7, 16, 1 << 19)])
def test_fewer_even_ranges_than_the_contexts_need_are_refused(max_splits, page, max_context):
    # a range of that many keys spans more pages than a workgroup keeps the ids of, whatever the rule's own width is
    wide = 2048 * 256 // 8
    assert StepContext.even_ranges(max_context, 256, 8, wide) > max_splits
    assert fused_entry(1, 8, 128, page, wide, max_splits, 256, max_context) == -3
    assert fused_entry(1, 8, 128, page, wide, max_splits, 256, 1 << 25) == -2


@pytest.mark.gpu
@pytest.mark.parametrize("q_heads,kv_heads,d,page,lengths,window", [
    (16, 8, 128, 16, [1, 2, 33, 64, 65, 66, 1000], None),
    (16, 8, 128, 16, [4931], None),
    (16, 1, 64, 32, [129, 700, 3], None),
    (5, 1, 128, 64, [2049, 1], 130),
    (16, 1, 256, 16, [300, 65], None),
    (3, 3, 192, 16, [90, 1100], 64),
    # beyond a share's width: two and three shares of workgroups a token; a window of them
    (16, 8, 128, 16, [9000, 4097, 4096, 7, 130, 1, 64, 500, 33, 2, 3000, 4161, 90, 17, 250, 8193], None),
    (8, 8, 64, 32, [9000, 4200, 1, 2, 3, 4, 5, 6, 7, 8, 9, 10, 11, 12, 13, 14], 8200),
    # more than 64 ranges, and more than 128, which the merge reads in several rounds
    (16, 1, 64, 32, [20011], None),
    (5, 1, 128, 16, [40000], None),
    (5, 1, 64, 64, [36000, 300], None),
])
def test_even_ranges_give_the_plain_attention_on_every_launch(q_heads, kv_heads, d, page, lengths, window):
    from test_kernels_gpu import kernels, plain_attention, tol
    k, dtype = kernels(torch.bfloat16), torch.bfloat16
    gen = torch.Generator().manual_seed(7)
    n, most = len(lengths), max(lengths)
    blocks = [-(-L // page) for L in lengths]
    perm = torch.randperm(sum(blocks), generator=gen)
    table = torch.full((n, max(blocks)), -1, dtype=torch.int32)
    k_pages = torch.full((sum(blocks), kv_heads, page, d), float("nan"), dtype=dtype)
    v_pages = torch.full((sum(blocks), kv_heads, d, page), float("nan"), dtype=dtype)
    keys, values, at = [], [], 0
    for s, L in enumerate(lengths):
        kk, vv = torch.randn((2, L - 1, kv_heads, d), generator=gen).to(dtype)
        keys.append(kk)
        values.append(vv)
        for b in range(blocks[s]):
            table[s, b] = perm[at]
            part = slice(b * page, min(L - 1, (b + 1) * page))
            k_pages[perm[at], :, :max(0, part.stop - part.start)] = kk[part].transpose(0, 1)
            v_pages[perm[at], :, :, :max(0, part.stop - part.start)] = vv[part].permute(1, 2, 0)
            at += 1
    qkv = (torch.randn((n, (q_heads + 2 * kv_heads) * d), generator=gen) * 1.5).to(dtype)
    units, workgroups = n * kv_heads, 256
    wide = -(-2048 * workgroups // units // 64) * 64
    splits = StepContext.even_ranges(2 * most, workgroups, units, wide)      # (laid out for more than the longest, as a graph's bucket is)
    partial = torch.full((k.attention_partial_numel(n, q_heads, d, splits),), float("nan"), device="cuda")
    arrivals = torch.zeros(units, dtype=torch.int32, device="cuda")
    rows = torch.arange(n, dtype=torch.int32, device="cuda")
    pos = torch.tensor([L - 1 for L in lengths], dtype=torch.int32, device="cuda")
    first = None
    for _ in range(3):                                     # the counters are there for the next launch
        kp, vp = k_pages.cuda(), v_pages.cuda()
        out = torch.full((n, q_heads * d), float("nan"), dtype=dtype, device="cuda")
        k.attention_decode_fused(qkv.cuda(), kp, vp, table.cuda(), rows, pos, out, rows, torch.ones_like(rows), n, q_heads, kv_heads, d, page,
                                 1 / math.sqrt(d), None, None, 0.0, None, partial, window=window, split_keys=wide, max_splits=splits,
                                 arrivals=arrivals, workgroups=workgroups)
        assert arrivals.eq(0).all()
        assert first is None or torch.equal(out, first)    # whoever merges, the sums' order is the ranges'
        first = out
    own_k = qkv[:, q_heads * d:(q_heads + kv_heads) * d].view(n, 1, kv_heads, d)
    own_v = qkv[:, (q_heads + kv_heads) * d:].view(n, 1, kv_heads, d)
    for s, L in enumerate(lengths):
        want = plain_attention(qkv[s, :q_heads * d].double().view(q_heads, d), torch.cat([keys[s], own_k[s]]).double(),
                               torch.cat([values[s], own_v[s]]).double(), 1 / math.sqrt(d), window)
        torch.testing.assert_close(first[s].double().cpu().view(q_heads, d), want, **tol(dtype))
        pg = table[s, (L - 1) // page]
        assert torch.equal(kp[pg, :, (L - 1) % page].cpu(), own_k[s, 0]) and torch.equal(vp[pg, :, :, (L - 1) % page].cpu(), own_v[s, 0])


@pytest.mark.gpu
def test_one_range_a_token_needs_no_room_for_results():
    # (one workgroup has all of a token's keys: its sums stay in LDS)
    from test_kernels_gpu import kernels
    k = kernels(torch.bfloat16)
    gen = torch.Generator().manual_seed(3)
    draw = lambda *shape: torch.randn(shape, generator=gen).bfloat16().cuda()
    table = torch.arange(24, dtype=torch.int32, device="cuda").view(3, 8)
    pages, qkv = (draw(24, 2, 16, 64), draw(24, 2, 64, 16)), draw(3, 8 * 64)
    rows, pos = torch.arange(3, dtype=torch.int32, device="cuda"), torch.tensor([0, 40, 127], dtype=torch.int32, device="cuda")
    outs = []
    for workgroups, room in ((0, torch.full((k.attention_partial_numel(3, 4, 64, 1),), float("nan"), device="cuda")), (0, None), (6, None)):
        out = torch.full((3, 256), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.attention_decode_fused(qkv, pages[0].clone(), pages[1].clone(), table, rows, pos, out, rows, torch.ones_like(rows), 3, 4, 2, 64, 16, 0.125,
                                 None, None, 0.0, None, room, split_keys=128 if workgroups else 0, workgroups=workgroups)
        outs.append(out)
        assert room is None or torch.isnan(room).all()
    assert torch.isfinite(outs[0]).all() and all(torch.equal(o, outs[0]) for o in outs[1:])
    with pytest.raises(KernelError):
        k.attention_decode_fused(qkv, *pages, table, rows, pos, out, rows, torch.ones_like(rows), 3, 4, 2, 64, 16, 0.125, None, None, 0.0, None, None,
                                 split_keys=64, max_splits=2)
