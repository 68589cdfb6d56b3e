"""Products of experts with few rows each on narrow tiles: the bits of the kernel that stages through registers."""
import ctypes

import pytest
import torch

pytestmark = pytest.mark.gpu


# (experts without rows, with one, with exactly a tile's, one more, far more than the average; fewer blocks of k than the LDS holds;
# columns that end inside a tile; averages on both sides of every line of the rule)
@pytest.mark.parametrize("counts", [[1], [0, 3, 0, 32, 33, 1], [64, 0, 65, 5], [20, 20, 20], [20, 21, 20], [55, 56, 55, 57, 56], [56, 57, 56, 55, 56],
                                    [200, 0, 0, 0, 0, 0, 0, 0, 0, 0, 0, 1], [0, 0, 0]])
@pytest.mark.parametrize("n,k,act", [(128, 64, None), (352, 192, "relu_squared"), (160, 640, "gated_silu"), (1056, 1024, "gated_clamped"), (136, 448, "gelu_erf")])
def test_bits_do_not_turn_on_the_tile(counts, n, k, act):
    from mini_llm_runtime_amd.kernels.ops import Kernels
    kernels = Kernels(torch.bfloat16)
    lib = kernels._lib("grouped_gemm")
    gen = torch.Generator("cuda").manual_seed(n + k)
    experts, rows, tokens = len(counts), max(1, sum(counts)), 77
    x = torch.randn(tokens, k, generator=gen, device="cuda").to(torch.bfloat16)
    w = (torch.randn(experts, n, k, generator=gen, device="cuda") * k ** -0.5).to(torch.bfloat16)
    gather = torch.randint(0, tokens, (rows,), generator=gen, device="cuda", dtype=torch.int32)
    offsets = torch.tensor([sum(counts[:i]) for i in range(experts + 1)], dtype=torch.int32, device="cuda")
    gated = act is not None and act.startswith("gated")
    limits = dict(limit=0.7, slope=1.5) if act == "gated_clamped" else {}

    def product(rows_of):
        out = torch.full((rows, n // 2 if gated else n), float("nan"), dtype=torch.bfloat16, device="cuda")
        kernels.experts_gemm(rows_of, w, out, offsets, gather=gather, act=act, **limits)
        return out.view(torch.int16)
    off = torch.empty(tokens * k + 1, dtype=torch.bfloat16, device="cuda")[1:].view(tokens, k)       # (off 16 bytes: the other kernel's)
    off.copy_(x)
    want = product(off)
    assert torch.equal(product(x), want)
    if act not in ("gated_clamped", None, "gelu_erf"):
        p, i = (lambda t: ctypes.c_void_p(t.data_ptr())), ctypes.c_int
        for shape in range(6):
            out = torch.full((rows, n // 2 if gated else n), float("nan"), dtype=torch.bfloat16, device="cuda")
            assert lib.mlr_experts_wide(p(x), p(w), p(out), p(offsets), p(gather), i(rows), i(n), i(k), i(experts), i(kernels.GROUPED_ACTS[act]),
                                        i(shape), ctypes.c_long(tokens), ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)) == 0
            assert torch.equal(out.view(torch.int16), want), shape
