"""The norms that keep a row in registers, at the widths where a thread takes one piece more, and beyond those that are kept."""
import pytest
import torch

pytestmark = pytest.mark.gpu
# one rounding to bfloat16 (half an ulp: 2^-9 of the value) of a 32-bit result whose own error is far below it
CLOSE = dict(rtol=2 ** -8, atol=1e-5)


def rows(n, width, seed):
    gen = torch.Generator().manual_seed(seed)
    return lambda *shape: torch.randn(*(shape or (n, width)), generator=gen).cuda()


@pytest.mark.parametrize("width", [8, 504, 512, 520, 1024, 1032, 1536, 2048, 2056, 4096, 4104, 6144, 6152, 8200])
@pytest.mark.parametrize("n", [3, 70])
def test_rows_of_every_number_of_pieces(n, width):
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16)
    draw = rows(n, width, n + width)
    h, d1, d2, w1, w2 = draw(), draw().bfloat16(), draw().bfloat16(), draw(width), draw(width)
    empty = lambda: torch.full((n, width), float("nan"), dtype=torch.bfloat16, device="cuda")
    rms = lambda x: x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5)
    for write_h in (True, False):
        got, out = h.clone(), empty()
        k.add_rmsnorm(got, d1, w1, out, 1e-5, write_h=write_h)
        x = h + d1.float()
        torch.testing.assert_close(out.float(), rms(x) * w1, **CLOSE)
        assert torch.equal(got, x if write_h else h)
    got, out, other = h.clone(), empty(), empty()
    k.add2_rmsnorm2(got, d1, d2, w1, w2, out, other, 1e-5)
    x = h + (d1.float() + d2.float())
    assert torch.equal(got, x)
    torch.testing.assert_close(out.float(), rms(x) * w1, **CLOSE)
    torch.testing.assert_close(other.float(), rms(x) * w2, **CLOSE)
    got, out = h.clone(), empty()
    k.add2_layernorm(got, d1, d2, w1, w2, out, 1e-5)
    assert torch.equal(got, x)
    want = torch.nn.functional.layer_norm(x, (width,), w1, w2, 1e-5)
    torch.testing.assert_close(out.float(), want, **CLOSE)
    if width <= 4096:
        got, cast = h.clone(), empty()
        k.layernorm_add(d1, w1, w2, got, cast=cast, eps=1e-5)
        want = h + torch.nn.functional.layer_norm(d1.float(), (width,), w1, w2, 1e-5)
        torch.testing.assert_close(got, want, rtol=1e-5, atol=2e-5)        # (32-bit sums of up to 4096 values)
        assert torch.equal(cast, got.bfloat16())


@pytest.mark.parametrize("part,parts", [(8, 5), (512, 2), (520, 1), (1024, 2), (1032, 1), (2048, 1), (2056, 2), (4096, 1), (4104, 1), (8192, 1)])
@pytest.mark.parametrize("gate_first", [True, False])
def test_parts_of_every_number_of_pieces(part, parts, gate_first):
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16)
    n, width = 7, part * parts
    draw = rows(n, width, part + parts)
    y, gate, w = draw(), draw().bfloat16(), draw(part)
    out = torch.full((n, width), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gated_part_norm(y, gate, w, out, part, 1e-5, gate_first)
    g = torch.nn.functional.silu(gate.float())
    x = (y * g if gate_first else y).view(n, parts, part)
    want = (x / torch.sqrt((x * x).mean(-1, keepdim=True) + 1e-5) * w).reshape(n, width) * (1.0 if gate_first else g)
    torch.testing.assert_close(out.float(), want, **CLOSE)
