"""Products of up to 16 rows in the many-row kernel's narrow tiles: when they are taken, and their bits."""
import ctypes

import pytest
import torch

from mini_llm_runtime_amd.kernels import Kernels
from mini_llm_runtime_amd.kernels import ops


def without_gpu(routed=False):
    k = object.__new__(Kernels)
    k.dtype, k.library_gemm, k.routed, k.profiler = torch.bfloat16, True, routed, None
    k._libs, k._wide_choices, k._split = {}, {}, None
    return k


@pytest.mark.parametrize("rows,columns,inner,gated,taken", [
    (1, 2048, 2048, False, True), (16, 2048, 1408, False, True), (17, 2048, 2048, False, False), (8, 2048, 1344, False, False),
    (8, 4352, 1024, False, False), (8, 4353, 1024, False, True), (8, 383, 2048, False, False), (8, 384, 2048, False, True),
    (8, 16385, 2048, False, False), (8, 2048, 6144, False, True), (8, 2048, 6208, False, False), (8, 2048, 2050, False, False),
    (8, 704, 1024, True, True), (8, 704, 960, True, False), (8, 16384, 3072, True, True), (8, 8193, 3136, True, False),
    # (many columns: not where the rows of a tile lie on the same channels of memory, nor with a short k or few rows)
    (8, 6656, 2048, True, True), (8, 6657, 2048, True, False), (8, 16384, 2048, True, False), (16, 8192, 4096, True, False), (1, 7168, 1536, True, False),
    (1, 7168, 1792, True, True), (7, 10240, 2560, True, True), (7, 10241, 2560, True, False), (8, 10241, 2560, True, True), (8, 8192, 3136, True, True),
    (8, 8192, 2048, False, True), (8, 8193, 2560, False, False), (9, 8193, 2560, False, True), (1, 12800, 2560, False, False),
    (1, 12801, 2560, False, True), (1, 16384, 4096, False, False), (9, 16384, 4096, False, True)])
def test_few_rows_of_a_long_enough_inner_size(rows, columns, inner, gated, taken):
    for routed in (False, True):
        assert without_gpu(routed).narrow_product(rows, columns, inner, gated) == taken


@pytest.mark.gpu
@pytest.mark.parametrize("columns,inner,gated", [(384, 1408, False), (2050, 1984, False), (4360, 1024, False), (1001, 2112, False), (8192, 6144, False),
                                                 (704, 1024, True), (1000, 1088, True), (5632, 2048, True), (385, 3136, True)])
@pytest.mark.parametrize("rows", [1, 7, 16])
def test_narrow_tiles_have_the_bits_of_the_streaming_kernel(rows, columns, inner, gated):
    k = Kernels(torch.bfloat16)
    assert k.narrow_product(rows, columns, inner, gated)
    gen = torch.Generator().manual_seed(rows + columns + inner)
    draw = lambda *shape: torch.randn(*shape, generator=gen).to(torch.bfloat16).cuda()
    a, w = draw(rows, inner), draw(columns * (2 if gated else 1), inner)
    want, got = (torch.full((rows, columns), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    place = lambda t: ctypes.c_void_p(t.data_ptr())
    sizes = [ctypes.c_int(n) for n in (rows, columns, inner)]
    lib = k._lib("gemm")
    if gated:
        assert lib.mlr_gemm_gated_silu(place(a), place(w), place(want), *sizes, ops._stream()) == 0
        k.gemm_gated_silu(a, w, got)
    else:
        assert lib.mlr_gemm(place(a), place(w), place(want), *sizes, ctypes.c_int(0), ops._stream()) == 0
        k.gemm(a, w, got)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))


# (columns whose address is not on 16 bytes go to the streaming kernel: its bits)
@pytest.mark.gpu
@pytest.mark.parametrize("columns,inner", [(704, 1024), (1000, 1088), (5632, 2048), (3000, 2112)])
@pytest.mark.parametrize("rows", [1, 7, 16, 17, 32, 64])
def test_a_clamped_gate_in_narrow_tiles_has_the_bits_of_the_streaming_kernel(columns, inner, rows):
    k = Kernels(torch.bfloat16)
    gen = torch.Generator().manual_seed(rows + columns + inner)
    a = torch.randn(rows, inner, generator=gen).to(torch.bfloat16).cuda()
    room = torch.empty(2 * columns * inner + 4, dtype=torch.bfloat16, device="cuda")
    w, off = room[:-4].view(2 * columns, inner), room[4:].view(2 * columns, inner)
    values = (0.1 * torch.randn(2 * columns, inner, generator=gen)).to(torch.bfloat16).cuda()
    want, got = (torch.full((rows, columns), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    w.copy_(values)
    k.gemm_gated_clamped(a, w, got, 2.0, 1.7)
    off.copy_(values)
    k.gemm_gated_clamped(a, off, want, 2.0, 1.7)
    assert torch.equal(got.view(torch.int16), want.view(torch.int16))
