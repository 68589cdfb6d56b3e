"""The product of attention's q, k and v with the heads' epilogue (`Kernels.gemm_qkv`): the bits of the product followed by
`qk_norm_rope_kv`, at the edges of its tiles, of pages and of requests."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu

HEAD = 128


def case(hq, hkv, k, page, counts, starts, seed):
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    m, n_req = sum(counts), len(counts)
    positions = torch.cat([torch.arange(s, s + n) for s, n in zip(starts, counts)]).to(torch.int32).cuda()
    slots = torch.cat([torch.full((n,), i) for i, n in enumerate(counts)]).to(torch.int32).cuda()
    most = max(s + n for s, n in zip(starts, counts))
    blocks = -(-most // page)
    table = torch.randperm(n_req * blocks, generator=torch.Generator().manual_seed(seed)).to(torch.int32).view(n_req, blocks)
    x = rnd(m, k).to(torch.bfloat16)
    w = (rnd((hq + 2 * hkv) * HEAD, k) * k ** -0.5).to(torch.bfloat16)
    norms = (rnd(HEAD) + 1.0, rnd(HEAD) + 1.0)
    angle = torch.arange(most, device="cuda")[:, None] * 10000.0 ** (-torch.arange(HEAD // 2, device="cuda") / (HEAD // 2))
    rope = torch.cat([torch.cos(angle), torch.sin(angle)], 1).float().contiguous()
    return x, w, positions, slots, table.contiguous().cuda(), norms, rope, n_req * blocks


def run(k, fused, x, w, positions, slots, table, norms, rope, pages, hq, hkv, page, write, shape):
    kp = torch.full((pages, hkv, page, HEAD), float("nan"), dtype=torch.bfloat16, device="cuda")
    vp = torch.full((pages, hkv, HEAD, page), float("nan"), dtype=torch.bfloat16, device="cuda")
    q = torch.full((x.shape[0], hq * HEAD), float("nan"), dtype=torch.bfloat16, device="cuda")
    if fused:
        k.gemm_qkv(x, w, q, kp, vp, table, slots, positions, *norms, 1e-6, rope, hq, hkv, HEAD, page, write, shape=shape)
    else:
        qkv = torch.empty((x.shape[0], w.shape[0]), dtype=torch.bfloat16, device="cuda")
        stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
        assert k._lib("gemm").mlr_gemm_wide(*(ctypes.c_void_p(t.data_ptr()) for t in (x, w, qkv)), x.shape[0], w.shape[0], x.shape[1],
                                            0, -1, 0, stream) == 0
        k.qk_norm_rope_kv(qkv, q, kp, vp, table, slots, positions, *norms, 1e-6, rope, hq, hkv, HEAD, page, write)
    return [t.view(torch.int16) for t in (q, kp, vp)]


# (one head short of a tile of two, a tile of queries, keys and values; rows one beyond a tile and far from it; k of fewer blocks
# than the LDS holds; portions from inside a page, from an odd place, behind single tokens; pages of 8 and of 48)
@pytest.mark.parametrize("sizes", [(3, 2, 64, 16, [65], [0]), (2, 1, 192, 16, [1, 1, 1, 127], [5, 31, 16, 3]),
                                   (4, 2, 256, 8, [257, 130], [8, 1]), (5, 1, 1024, 48, [96, 97], [40, 0]),
                                   (1, 1, 128, 16, [300], [7]), (16, 8, 1024, 16, 32 * [1] + [480], list(range(32)) + [0])])
@pytest.mark.parametrize("shape", [-1, 4, 5, 7, 9])
def test_bits_of_the_two_launches(sizes, shape):
    from mini_llm_runtime_amd.kernels.ops import Kernels
    hq, hkv, inner, page, counts, starts = sizes
    k = Kernels(torch.bfloat16)
    made = case(hq, hkv, inner, page, counts, starts, 5)
    x, w, positions, slots, table, norms, rope, pages = made
    for write, normed in ((True, True), (True, False), (False, True)):
        args = (x, w, positions, slots, table, norms if normed else (None, None), rope, pages, hq, hkv, page, write, shape)
        for got, want in zip(run(k, True, *args), run(k, False, *args)):
            assert torch.equal(got, want)


def test_missing_pages_and_places_beyond_the_table():
    """A page that is not there and a position beyond the request's row of the table: nothing is written for them."""
    from mini_llm_runtime_amd.kernels.ops import Kernels
    hq, hkv, page = 2, 2, 16
    k = Kernels(torch.bfloat16)
    x, w, positions, slots, table, norms, rope, pages = case(hq, hkv, 128, page, [100, 60], [0, 20], 6)
    table[0, 2] = -1
    short = table[:, :4].contiguous()
    for shape in (4, 5, 7, 9):
        args = (x, w, positions, slots, short, norms, rope, pages, hq, hkv, page, True, shape)
        for got, want in zip(run(k, True, *args), run(k, False, *args)):
            assert torch.equal(got, want)


def test_the_choice():
    """Sizes that are not this form's keep the two launches, and what it refuses it refuses loudly."""
    from mini_llm_runtime_amd.kernels.ops import KernelError, Kernels
    k = Kernels(torch.bfloat16)
    assert k.qkv_product(2048, 16, 8, 128, 1024, 16) and k.qkv_product(512, 16, 8, 128, 1024, 16)
    assert not k.qkv_product(64, 16, 8, 128, 1024, 16) and not k.qkv_product(2048, 16, 8, 64, 1024, 16)
    assert not k.qkv_product(2048, 16, 8, 128, 1000, 16) and not k.qkv_product(2048, 16, 8, 128, 1024, 20)
    odd = torch.empty(2049, dtype=torch.bfloat16, device="cuda")[1:]
    assert not k.qkv_product(2048, 16, 8, 128, 1024, 16, odd)
    x, w, positions, slots, table, norms, rope, pages = case(2, 1, 128, 16, [70], [0], 7)
    with pytest.raises(KernelError):
        run(k, True, x, w, positions, slots, table, norms, rope[:, :64].contiguous(), pages, 2, 1, 16, True, -1)
