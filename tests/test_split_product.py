"""Products of up to 64 rows whose tiles several workgroups share: when they are taken, and their bits."""
import ctypes

import pytest
import torch

from mini_llm_runtime_amd.kernels import Kernels
from mini_llm_runtime_amd.kernels import ops


def without_gpu(routed=False):
    k = object.__new__(Kernels)
    k.dtype, k.library_gemm, k.routed, k.profiler = torch.bfloat16, True, routed, None
    k._libs, k._wide_choices, k._split, k._split_stream = {}, {}, None, None
    return k


@pytest.mark.parametrize("rows,columns,inner,taken", [
    (1, 2048, 5632, True), (16, 2048, 3584, True), (16, 2048, 3520, False), (8, 4096, 4096, False), (8, 4096, 5120, True), (8, 8192, 3584, True),
    (8, 8193, 9216, False), (16, 4096, 12288, True), (17, 4096, 12288, True), (64, 4096, 12288, True), (65, 4096, 12288, False), (64, 4096, 2048, False),
    (64, 2048, 2560, True), (32, 2048, 2560, False), (64, 1024, 2560, False), (32, 2048, 3136, True), (32, 2049, 3136, False),
    (33, 4096, 3136, True), (20, 4097, 4224, False), (64, 6144, 6144, True), (64, 8192, 9216, True), (64, 16384, 14336, True),
    (64, 16385, 14336, False), (64, 4096, 12289, False),
    # (inner sizes that put the rows of weight on the same channels of memory, few rows, round sizes that the library cuts itself)
    (16, 2560, 8192, True), (16, 2561, 8192, False), (8, 4096, 24576, False), (8, 4096, 16384, True), (16, 4097, 12288, False), (16, 4097, 12352, True),
    (4, 3073, 8960, False), (5, 3073, 8960, True), (1, 3072, 8960, True), (1, 3073, 14336, True), (20, 3072, 8192, True), (20, 3073, 8192, False),
    (48, 4096, 8192, True), (48, 4097, 8192, False), (32, 6144, 12288, True), (32, 6145, 12288, False), (48, 8192, 12288, True), (32, 4097, 24576, False),
    (48, 6144, 24576, True), (64, 8192, 16384, False), (64, 8193, 16384, False), (64, 10240, 15424, True), (64, 10240, 15360, False),
    (64, 11265, 15424, False), (64, 12288, 14336, False), (32, 12288, 14336, True), (24, 4096, 7168, False), (25, 4096, 7168, True), (24, 3072, 5056, False),
    (24, 3072, 5120, True), (24, 2048, 4224, True), (33, 1024, 5120, False), (33, 1024, 5184, True), (32, 1024, 5120, True)])
def test_long_inner_sizes_of_few_rows_are_shared_out(rows, columns, inner, taken):
    assert without_gpu().split_product(rows, columns, inner) == taken
    assert without_gpu(routed=True).split_product(rows, columns, inner) == (taken and rows <= 16)


@pytest.mark.parametrize("rows,columns,inner,shared", [
    (8, 2048, 5632, True), (8, 2560, 5120, True), (8, 2561, 5120, False), (8, 8192, 3584, False), (8, 4096, 6144, False), (8, 5120, 6144, False),
    (8, 5121, 6144, True), (8, 4096, 6208, True), (17, 2048, 5632, True), (17, 4096, 12288, True), (32, 4096, 5120, True)])
def test_narrow_tiles_come_before_shared_ones_over_many_columns(monkeypatch, rows, columns, inner, shared):
    k = without_gpu()
    monkeypatch.setattr(ops, "_stream", lambda: ctypes.c_void_p(0))
    k._split, k._split_stream = ("room", "counters"), 0
    assert k.shares_tiles(rows, columns, inner) == shared


def test_only_the_stream_that_has_the_room_shares_tiles(monkeypatch):
    k, now = without_gpu(), [0]
    monkeypatch.setattr(ops, "_stream", lambda: ctypes.c_void_p(now[0]))
    assert not k.shares_tiles(8, 2048, 5632) and not k.has_split()               # (no room at all)
    k.claim_split()
    k._split = ("room", "counters")
    assert not k.has_split()                               # (nobody has it yet)
    for owner in (0, 4096, 0):
        now[0] = owner
        k.claim_split()
        for stream in (0, 4096, 8192):
            now[0] = stream
            assert k.shares_tiles(8, 2048, 5632) and k.has_split() == (stream == owner)


# (inner sizes whose last share is one block, a part's last block missing, as many as parts; columns in whole tiles, ragged, odd)
@pytest.mark.gpu
@pytest.mark.parametrize("inner", [512, 448, 64 * 25, 64 * 49, 4096, 64 * 67])
@pytest.mark.parametrize("rows,columns", [(1, 64), (5, 40), (16, 1000), (16, 2050), (17, 16), (32, 64), (31, 1000), (33, 129), (64, 128), (50, 2047), (64, 4096)])
def test_a_shared_tile_has_the_bits_of_one_workgroups(rows, columns, inner):
    k = Kernels(torch.bfloat16)
    gen = torch.Generator().manual_seed(rows + columns + inner)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()
    a, w = draw(rows, inner), draw(columns, inner)
    want = torch.empty(rows, columns, dtype=torch.bfloat16, device="cuda")
    number, place = ctypes.c_int, lambda t: ctypes.c_void_p(t.data_ptr())
    lib, stream = k._lib("gemm"), ops._stream()
    sizes = (number(rows), number(columns), number(inner))
    if rows > 16:
        assert lib.mlr_gemm_wide(place(a), place(w), place(want), *sizes, number(0), number(-2), number(0), stream) == 0
    else:
        assert lib.mlr_gemm(place(a), place(w), place(want), *sizes, number(0), stream) == 0
    partial = torch.full((1 << 23,), float("nan"), device="cuda")
    arrivals = torch.zeros(ops.SPLIT_COUNTERS, dtype=torch.int32, device="cuda")
    taken = 0
    for shape in range(-1, 10):
        for _ in range(2):                               # (the counters are what they were)
            got = torch.full_like(want, float("nan"))
            code = lib.mlr_gemm_split(place(a), place(w), place(got), *sizes, place(partial), ctypes.c_long(partial.numel()), place(arrivals),
                                      number(arrivals.numel()), number(shape), stream)
            if code == -1:
                assert torch.isnan(got).all()            # (too few blocks of k for the shares: nothing was launched)
                continue
            assert code == 0 and torch.equal(got.view(torch.int16), want.view(torch.int16)), shape
            taken += 1
        assert not arrivals.any()
    assert taken >= (0 if inner < 512 else 8)
    # no room, no launch
    code = lib.mlr_gemm_split(place(a), place(w), place(got), *sizes, place(partial), ctypes.c_long(64), place(arrivals),
                              number(arrivals.numel()), number(-1), stream)
    assert code == -1


@pytest.mark.gpu
def test_the_runners_kernels_share_products_out_and_others_do_not():
    k, other = Kernels(torch.bfloat16), Kernels(torch.bfloat16)
    k.reserve_split_workspace("cuda")
    a, w = torch.randn(40, 4160, device="cuda").bfloat16(), torch.randn(1500, 4160, device="cuda").bfloat16()
    out, again = (torch.empty(40, 1500, dtype=torch.bfloat16, device="cuda") for _ in range(2))
    k.gemm(a, w, out)
    few = torch.empty_like(out)
    assert k._lib("gemm").mlr_gemm_wide(*(ctypes.c_void_p(t.data_ptr()) for t in (a, w, few)), *(ctypes.c_int(n) for n in (40, 1500, 4160, 0, -2, 0)),
                                        ops._stream()) == 0
    assert torch.equal(out.view(torch.int16), few.view(torch.int16)) and other._split is None
    other.gemm(a, w, again)
    want = a.float() @ w.float().T
    for got in (out, again):                             # (one rounding to bfloat16 of sums whose terms are about 1)
        torch.testing.assert_close(got.float(), want, rtol=2 ** -8, atol=2 ** -8)
    # between a product of the library, which has the rest of the scratch memory, and another
    k.gemm(torch.randn(64, 2048, device="cuda").bfloat16(), torch.randn(4096, 2048, device="cuda").bfloat16(),
           torch.empty(64, 4096, device="cuda"))
    k.gemm(a, w, again)
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))


# a long product on the stream that has the room, another beside it on a second stream and in a capture of the caller's own: the
# same bits everywhere, whoever shares
@pytest.mark.gpu
@pytest.mark.parametrize("rows", [16, 40])
def test_products_of_two_streams_at_once_do_not_meet(rows):
    k = Kernels(torch.bfloat16)
    k.reserve_split_workspace("cuda")
    gen = torch.Generator().manual_seed(5)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()
    a, w = [draw(rows, 5632) for _ in range(2)], [draw(2048, 5632) for _ in range(2)]
    want = [torch.empty(rows, 2048, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
    assert k.shares_tiles(rows, 2048, 5632) and k.has_split()
    for i in range(2):
        k.gemm(a[i], w[i], want[i])
    outs = [[torch.full_like(want[i], float("nan")) for _ in range(20)] for i in range(2)]
    other, graph, captured = torch.cuda.Stream(), torch.cuda.CUDAGraph(), torch.full_like(want[1], float("nan"))
    torch.cuda.synchronize()
    with torch.cuda.graph(graph):
        assert not k.has_split()
        k.gemm(a[1], w[1], captured)
    for n in range(20):
        k.gemm(a[0], w[0], outs[0][n])
        with torch.cuda.stream(other):
            assert not k.has_split()
            k.gemm(a[1], w[1], outs[1][n])
            graph.replay()
    torch.cuda.synchronize()
    same = lambda x, y: torch.equal(x.view(torch.int16), y.view(torch.int16))
    assert same(captured, want[1]) and all(same(out, want[i]) for i in range(2) for out in outs[i])
    assert not k._split[1].any()
