"""Row kernels that take several values an access against the same kernels one value at a time (reached by an operand that
does not start on 16 bytes): the same arithmetic, so the same results."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def kernels(dtype):
    from mini_llm_runtime_amd.kernels import Kernels
    return Kernels(dtype)


def moved(x):
    """The same values, one element behind an aligned start."""
    whole = torch.empty(x.numel() + 1, dtype=x.dtype, device=x.device)
    whole[1:] = x.flatten()
    return whole[1:].view(x.shape)


def ints(x):
    return torch.tensor(x, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("rows,channels", [(768, 2048), (767, 2056), (769, 2048), (5959, 264), (153, 10288)])
def test_causal_conv_of_many_rows(rows, channels):
    k = kernels(torch.bfloat16)
    gen = torch.Generator("cuda").manual_seed(rows + channels)
    x = torch.randn(rows, channels, generator=gen, device="cuda").bfloat16()
    w = torch.randn(channels, 4, generator=gen, device="cuda")
    b = torch.randn(channels, generator=gen, device="cuda")
    offset = 3
    live = torch.randn(5, offset + 3 * channels, generator=gen, device="cuda")
    cut = [(1, 7, 1), (3, 0, 2), (0, 5, 9), (4, 40, rows - 12)]              # slot, first position, tokens
    slots = ints([s for s, p, n in cut for _ in range(n)])
    pos = ints([p + i for s, p, n in cut for i in range(n)])
    for bias in (b, None):
        for silu in (True, False):
            got = []
            for weight in (w, moved(w)):
                out, stage = torch.empty_like(x), live.clone()
                k.causal_conv(x, weight, bias, out, live, stage, offset, slots, pos, silu=silu)
                got.append((out, stage))
            assert torch.equal(got[0][0], got[1][0]) and torch.equal(got[0][1], got[1][1])
    assert torch.equal(got[0][1][2], live[2])                                # (a slot without tokens)


@pytest.mark.parametrize("rows,heads,kv_heads,dim", [(1, 2, 1, 64), (5, 3, 2, 128), (70, 16, 4, 128)])
def test_norm_behind_the_rotation(rows, heads, kv_heads, dim):
    k = kernels(torch.bfloat16)
    gen = torch.Generator("cuda").manual_seed(rows)
    page = 16
    blocks = -(-rows // page)
    proj = torch.randn(rows, (heads + 2 * kv_heads) * dim, generator=gen, device="cuda").bfloat16()
    bias = torch.randn(proj.shape[1], generator=gen, device="cuda")
    angles = torch.randn(rows, dim // 2, generator=gen, device="cuda")
    rope = torch.cat([angles.cos(), angles.sin()], dim=1)
    w = torch.rand(dim, generator=gen, device="cuda") + 0.5
    got = []
    for b in (bias, moved(bias)):
        q = torch.zeros(rows, heads * dim, dtype=torch.bfloat16, device="cuda")
        pages = [torch.zeros(blocks, kv_heads, page, dim, dtype=torch.bfloat16, device="cuda") for _ in range(2)]
        k.sink_qkv_prep(proj, b, q, *pages, ints([list(range(blocks))]), ints([0] * rows), ints(list(range(rows))), w, w.flip(0).contiguous(), 1e-5,
                        rope, heads, kv_heads, dim, dim, page, norm="after")
        got.append([q.float(), pages[0].float(), pages[1].float()])
    for a, b in zip(*got):
        # (the sum of squares is taken in another order: at most the last place of a bfloat16)
        torch.testing.assert_close(a, b, rtol=2 ** -7, atol=1e-6)
    assert torch.equal(got[0][2], got[1][2])


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 1028, 2048, 4096, 4100, 9000])
def test_layer_norm_of_wide_rows(dtype, width):
    k = kernels(dtype)
    gen = torch.Generator("cuda").manual_seed(width)
    rows = 3
    x = (torch.randn(rows, width, generator=gen, device="cuda") + 2).to(dtype)
    h0 = torch.randn(rows, width, generator=gen, device="cuda")
    w, b = (torch.randn(width, generator=gen, device="cuda") for _ in range(2))
    want = torch.nn.functional.layer_norm(x.double().cpu(), (width,), w.double().cpu(), b.double().cpu(), 1e-5)
    want = h0.double().cpu() + want
    for weight in (w, moved(w)):
        h, cast = h0.clone(), torch.empty_like(x)
        k.layernorm_add(x, weight, b, h, cast=cast, eps=1e-5)
        torch.testing.assert_close(h.double().cpu(), want, rtol=1e-5, atol=1e-5)
        assert torch.equal(cast, h.to(dtype))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("width", [4, 260, 1000, 1028, 2048, 4096, 4100])
def test_layer_norm_of_wide_rows_adds_up_in_the_same_order(dtype, width):
    """A router behind the norm turns on its last bits: four values an access and one give the same ones, added to the float
    stream, cast beside it, and as the final norm's rows."""
    k = kernels(dtype)
    gen = torch.Generator("cuda").manual_seed(width)
    rows = 70
    x = (torch.randn(rows, width, generator=gen, device="cuda") * 3 + 1).to(dtype)
    h0 = torch.randn(rows, width, generator=gen, device="cuda")
    w, b = (torch.randn(width, generator=gen, device="cuda") for _ in range(2))
    picked = ints([5, 0, 69, 33])
    for bias in (b, None):
        got = []
        for weight in (w, moved(w)):
            h, cast, out = h0.clone(), torch.empty_like(x), torch.empty(4, width, dtype=dtype, device="cuda")
            k.layernorm_add(x, weight, bias, h, cast=cast, eps=1e-5)
            k.layernorm_rows(h0, weight, bias, out, 1e-5, rows=picked)
            got.append((h, cast, out))
        assert all(torch.equal(a, b) for a, b in zip(*got))


@pytest.mark.parametrize("rows,heads,keys", [(1, 3, 7), (300, 8, 128), (2, 1100, 256)])
def test_decay_per_channel(rows, heads, keys):
    k = kernels(torch.bfloat16)
    gen = torch.Generator("cuda").manual_seed(rows)
    z = torch.randn(rows, heads * keys, generator=gen, device="cuda") * 4
    bias, a_log = torch.randn(heads * keys, generator=gen, device="cuda"), torch.randn(heads, generator=gen, device="cuda")
    out = torch.full_like(z, float("nan"))
    k.channel_log_decay(z, bias, a_log, out, heads, keys)
    want = -a_log.double().exp().repeat_interleave(keys) * torch.nn.functional.softplus(z.double() + bias.double(), threshold=100.0)
    torch.testing.assert_close(out.double(), want, rtol=2e-6, atol=1e-9)
