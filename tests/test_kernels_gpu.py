"""Each HIP kernel alone against a plain formula in float64, at sizes other than the tiny
models' (the reference tests each op against a host formula in the same way,
tests/cuda_ops_tests.cu:38-72)."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

DTYPES = [torch.float32, torch.bfloat16]


def tol(dtype):
    return dict(atol=2e-4, rtol=2e-4) if dtype == torch.float32 else dict(atol=2e-2, rtol=2e-2)


def kernels(dtype):
    from mini_llm_runtime_amd.kernels import Kernels
    return Kernels(dtype)


def sample(k, logits, temp, u, tokens, status):
    need_f, need_i = k.sample_scratch(logits.shape[0])
    k.sample(logits, temp, u, tokens, status, torch.empty(need_f, device="cuda"),
             torch.empty(need_i, dtype=torch.int32, device="cuda"))


def rnd(shape, dtype, seed, scale=1.0):
    g = torch.Generator().manual_seed(seed)
    return (scale * torch.randn(shape, generator=g)).to(dtype).cuda()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [1, 17, 76, 128, 1000, 3072])
def test_embed_gather(dtype, width):
    k = kernels(dtype)
    table = rnd((37, width), dtype, 1)
    ids = torch.tensor([0, 36, 5, 5, 17], dtype=torch.int32).cuda()
    h = torch.full((5, width), 7.0, device="cuda")
    k.embed_gather(ids, table, h)
    assert torch.equal(h, table.float()[ids.long()])


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [1, 17, 31, 32, 33, 128, 1024, 3072])
def test_add_rmsnorm(dtype, width):
    k = kernels(dtype)
    rows = 5
    h0 = rnd((rows, width), torch.float32, 2, 3.0)
    delta = rnd((rows, width), dtype, 3)
    w = rnd((width,), torch.float32, 4)
    eps = 1e-5
    x = h0.double() + delta.double()
    want = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double()
    # fused add: h is updated
    h = h0.clone()
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, delta, w, out, eps)
    torch.testing.assert_close(h.double(), x, atol=1e-6, rtol=1e-6)
    torch.testing.assert_close(out.double(), want, **tol(dtype))
    # gathered rows, h untouched
    h = h0.clone()
    idx = torch.tensor([4, 0, 4], dtype=torch.int32).cuda()
    out = torch.empty((3, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, delta, w, out, eps, rows=idx, write_h=False)
    assert torch.equal(h, h0)
    torch.testing.assert_close(out.double(), want[idx.long()], **tol(dtype))
    # no delta
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, None, w, out, eps)
    x = h0.double()
    torch.testing.assert_close(out.double(), x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double(),
                               **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width,repeat", [(257, 1), (256, 1), (256, 10)])
def test_rmsnorm_extremes(dtype, width, repeat):
    """Amplitudes from 0 to the largest float and an eps from the smallest to the largest
    (tests/cuda_ops_tests.cu:274-301): a row whose squares do not fit 32 bits is scaled by its largest element
    first, as the reference's kernel does for every row (src/minillm/cuda/ops.cu:87-126).  The widths and row
    counts reach each variant of the kernel (one workgroup a row, scalar or 16 bytes a thread; one wavefront a
    row from 64 rows on), with and without a delta that is still to be added."""
    k = kernels(dtype)
    top = float(np.finfo(np.float32).max)
    amps = [0.0, 1e-30, 1e-15, 1.0, 1e15, 1e30, top] * repeat
    h = torch.zeros((len(amps), width))
    for r, a in enumerate(amps):
        h[r, 0::3] = -a
        h[r, 1::3] = 0.5 * a
        h[r, 2::3] = 0.5 * a
    h = h.cuda()
    w = torch.ones(width, device="cuda")
    zero = torch.zeros((len(amps), width), dtype=dtype, device="cuda")
    for eps in (float(np.finfo(np.float32).smallest_subnormal), 1e-6, top):
        x = h.double()
        want = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps)
        for delta, write_h in ((None, True), (zero, True), (zero, False)):
            out = torch.full((len(amps), width), 7.0, dtype=dtype, device="cuda")
            k.add_rmsnorm(h.clone(), delta, w, out, eps, write_h=write_h)
            assert torch.isfinite(out.float()).all(), (eps, write_h)
            torch.testing.assert_close(out.double(), want, **tol(dtype))
    # an infinity or a NaN in a row gives a row of NaN, and only that row
    bad = h.clone()
    bad[3, 5], bad[4, 7] = float("inf"), float("nan")
    out = torch.empty((len(amps), width), dtype=dtype, device="cuda")
    k.add_rmsnorm(bad, None, w, out, 1e-6)
    assert torch.isnan(out[3].float()).all() and torch.isnan(out[4].float()).all()
    assert torch.isfinite(out[[0, 1, 2, 5, 6]].float()).all()


@pytest.mark.parametrize("dtype", DTYPES)
def test_silu_mul_and_residual(dtype):
    k = kernels(dtype)
    inter = 100
    gate_up = rnd((7, 2 * inter), dtype, 5, 3.0)
    gate_up[0, :9] = torch.tensor([0, 1, -1, 80, -80, 1e4, -1e4, 30, -30], dtype=dtype)
    act = torch.empty((7, inter), dtype=dtype, device="cuda")
    k.silu_mul(gate_up, act)
    g, u = gate_up.double()[:, :inter], gate_up.double()[:, inter:]
    want = g / (1 + torch.exp(-g)) * u
    assert torch.isfinite(act.float()).all()
    torch.testing.assert_close(act.double(), want, **tol(dtype))
    h0 = rnd((7, inter), torch.float32, 6)
    h = h0.clone()
    k.residual_add(h, act)
    torch.testing.assert_close(h, h0 + act.float())


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("mnk", [(7, 19, 33), (5, 37, 131), (1, 311, 80), (16, 64, 64), (17, 130, 100),
                                 (64, 200, 76), (65, 257, 256), (200, 300, 1024), (2, 2048, 1024),
                                 (33, 48, 520), (48, 1000, 264), (8, 6144, 1024), (129, 100, 40),
                                 (5, 40, 192), (11, 72, 4160), (16, 33, 1024), (9, 130, 3072), (2, 24, 8192), (16, 40, 4096), (40, 96, 4096), (24, 56, 2048),
                                 (130, 70, 128), (300, 520, 192), (257, 1030, 64), (1000, 90, 320), (66, 4100, 1024)])
def test_gemm(dtype, mnk):
    """Odd shapes as in the reference's GEMM test (tests/cuda_unit_tests.cu:207-209)."""
    from mini_llm_runtime_amd.kernels import Kernels
    m, n, kk = mnk
    a = rnd((m, kk), dtype, 7)
    w = rnd((n, kk), dtype, 8)
    want = a.double() @ w.double().T
    # the engine's choice (many rows of the bfloat16 engine go to the library) and the hand-written kernels alone
    for k in (kernels(dtype), Kernels(dtype, library_gemm=False)):
        for out_dtype in {dtype, torch.float32}:
            out = torch.full((m, n), float("nan"), dtype=out_dtype, device="cuda")
            k.gemm(a, w, out)
            t = dict(atol=1e-4 * math.sqrt(kk), rtol=1e-5) if out_dtype == torch.float32 else \
                dict(atol=2e-2 * math.sqrt(kk) / 4, rtol=2e-2)
            torch.testing.assert_close(out.double(), want, **t)


@pytest.mark.parametrize("mnk", [(8, 6144, 2048), (3, 6100, 2048), (16, 5120, 2112), (1, 10240, 2048), (5, 4100, 4096),
                                 (8, 6144, 4096), (2, 5120, 8192)])
def test_gemm_two_strips_a_workgroup(mnk):
    """Few rows and numbers of columns that would deal strips of 16 unevenly to the compute units: a workgroup
    then owns two strips side by side (24, 20, ... columns), the last workgroup fewer.  Plain and with the rows'
    scale of a norm that was handed over; rows stay independent of the batch."""
    m, n, kk = mnk
    k = kernels(torch.bfloat16)
    a = rnd((m, kk), torch.bfloat16, 17)
    w = rnd((n, kk), torch.bfloat16, 18)
    want = a.double() @ w.double().T
    for out_dtype in (torch.bfloat16, torch.float32):
        out = torch.full((m, n), float("nan"), dtype=out_dtype, device="cuda")
        k.gemm(a, w, out)
        t = dict(atol=1e-4 * math.sqrt(kk), rtol=1e-5) if out_dtype == torch.float32 else \
            dict(atol=2e-2 * math.sqrt(kk) / 4, rtol=2e-2)
        torch.testing.assert_close(out.double(), want, **t)
    one = torch.empty((1, n), dtype=torch.bfloat16, device="cuda")
    k.gemm(a[m - 1:].contiguous(), w, one)
    assert torch.equal(one[0], out.to(torch.bfloat16)[m - 1]) or out_dtype != torch.bfloat16
    full = torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    k.gemm(a, w, full)
    assert torch.equal(one[0], full[m - 1])
    ss = (torch.rand((m, k.handoff_parts(kk)), device="cuda") + 0.5).float()
    scaled = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_prenormed(a, ss, 1e-6, w, scaled)
    scale = 1.0 / torch.sqrt(ss.double().sum(dim=1) / kk + 1e-6)
    torch.testing.assert_close(scaled.double(), want * scale[:, None], atol=2e-2 * math.sqrt(kk) / 4, rtol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
def test_gemm_rows_do_not_depend_on_the_batch(dtype):
    """A row's result is the same bits whatever rows stand beside it.  The float kernel has one order of
    additions for every M; the bfloat16 engine has two (up to 64 rows k is cut into eight parts, above that it is one
    chain), so bits agree up to 64 rows and above, and differ by rounding across the two.  (k no multiple of 64: the next
    test has those.)"""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(dtype, library_gemm=False)
    a = rnd((200, 264), dtype, 9)
    w = rnd((150, 264), dtype, 10)

    def run(lo, hi):
        out = torch.empty((hi - lo, 150), dtype=dtype, device="cuda")
        k.gemm(a[lo:hi].contiguous(), w, out)
        return out
    full = run(0, 200)
    small = run(0, 64)
    for lo, hi in [(0, 1), (3, 20), (30, 64), (0, 33)]:
        assert torch.equal(run(lo, hi), small[lo:hi])
    for lo, hi in [(0, 130), (100, 200), (65, 135)]:
        assert torch.equal(run(lo, hi), full[lo:hi])
    if dtype == torch.float32:
        assert torch.equal(small, full[:64])
    else:
        torch.testing.assert_close(small.float(), full[:64].float(), atol=0.13, rtol=1e-2)   # one bfloat16 step at |x| ~ 16


@pytest.mark.parametrize("n,kk", [(150, 64), (96, 256), (1127, 1088), (3072, 1024), (704, 2048), (2112, 2816), (5000, 576), (1040, 4096)])
def test_gemm_rows_up_to_64_have_one_order_of_sums(n, kk):
    """Whole blocks of k: up to 16 rows are the few-row kernel's, 17 to 64 those of tiles that read their operands out of LDS where
    they are faster.  A row has the same bits alone and among any of them, plain and with gate and silu."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16, library_gemm=False)
    a, w = rnd((64, kk), torch.bfloat16, 94), rnd((2 * n, kk), torch.bfloat16, 95, 0.3)

    def run(lo, hi, gated):
        out = torch.full((hi - lo, n if gated else 2 * n), float("nan"), dtype=torch.bfloat16, device="cuda")
        (k.gemm_gated_silu if gated else k.gemm)(a[lo:hi].contiguous(), w, out)
        return out
    for gated in (False, True):
        alone = torch.cat([run(i, i + 1, gated) for i in range(64)])
        for lo, hi in [(0, 16), (48, 64), (0, 17), (20, 52), (7, 40), (0, 64)]:
            assert torch.equal(run(lo, hi, gated), alone[lo:hi]), (lo, hi, gated)


@pytest.mark.parametrize("n,kk", [(1, 4), (15, 1), (17, 60), (33, 64), (70, 511), (64, 516), (130, 528), (16400, 96), (4112, 1030), (96, 3072),
                                  (40, 12296)])
def test_gemm_float_edges(n, kk):
    """The float product at the edges of its row counts, strips, tiles and groups of k, rows that start on 16 bytes and rows that
    do not: one order of additions, so a row's bits are those it has alone; and every element well within the worst case of a
    chain over k, k 2^-24 sum |a w| (the roundings of a long chain go both ways: an eighth of that from k = 600 on)."""
    k = kernels(torch.float32)
    rows = 300 if n < 5000 else 70
    a, w = rnd((rows, kk), torch.float32, 21), rnd((n, kk), torch.float32, 22)
    a[3] *= 1e-20                                        # (products of row 3 below the smallest normal number)
    w[0] *= 1e-20

    def run(lo, hi):
        out = torch.full((hi - lo, n), float("nan"), device="cuda")
        k.gemm(a[lo:hi].contiguous(), w, out)
        return out
    whole = run(0, rows)
    bound = (max(kk / 8 + 16, 64) + 9) * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + kk * 2.0 ** -149
    assert bool(((whole.double() - a.double() @ w.double().T).abs() <= bound).all())
    for lo, hi in [(0, 1), (3, 4), (1, 9), (0, 9), (2, 18), (5, 22), (0, 32), (4, 37), (0, 64), (1, 66), (0, rows - 1)]:
        assert torch.equal(run(lo, hi), whole[lo:hi]), (lo, hi)
    shifted = torch.empty(rows * kk + 1, device="cuda")[1:].view(rows, kk).copy_(a)      # rows 4 bytes off
    out = torch.empty((rows, n), device="cuda")
    k.gemm(shifted, w, out)
    assert torch.equal(out, whole)


@pytest.mark.parametrize("m,n,kk", [(1, 16, 4), (1, 1, 1), (5, 40, 1028), (16, 33, 127), (9, 12400, 260), (33, 5200, 132), (70, 3300, 516),
                                    (32, 20000, 68), (130, 5000, 132), (2048, 4096, 36), (2048, 4090, 31)])
def test_gemm_float_is_one_chain_over_k(m, n, kk):
    """Every element of the float product is fmaf after fmaf from k = 0 up, to the bit, in every kernel and tile (a sampled token
    lies within the last bits of a product now and then, so the order is part of the result).  Factors are whole numbers below
    128 times 2^-3 .. 2^3: products and their sums up to 2^21 (k below 2^11) are whole multiples of 2^-6 and exact in 64 bits, so
    that rounding such a sum to 32 bits is what fmaf does."""
    k = kernels(torch.float32)
    g = torch.Generator("cuda").manual_seed(m + n + kk)

    def coarse(*shape):
        return torch.randint(-127, 128, shape, generator=g, device="cuda").float() * 2.0 ** torch.randint(-3, 4, shape, generator=g, device="cuda")
    a, w = coarse(m, kk), coarse(n, kk)
    want = torch.zeros((m, n), device="cuda")
    for i in range(kk):
        want = (want.double() + a[:, i, None].double() * w[None, :, i].double()).float()
    assert kk < 64 or not torch.equal(want, (a.double() @ w.double().T).float())      # (the chain's roundings are to be seen)
    shifted = torch.empty(m * kk + 1, device="cuda")[1:].view(m, kk).copy_(a)      # rows 4 bytes off
    for rows in (a, shifted):
        out = torch.full((m, n), float("nan"), device="cuda")
        k.gemm(rows, w, out)
        assert torch.equal(out, want)


@pytest.mark.parametrize("m,n,kk", [(1, 5, 4), (8, 3072, 1024), (16, 33, 60), (17, 100, 68), (5, 8192, 260), (40, 1500, 448), (33, 2600, 516)])
def test_gemm_gated_silu_float(m, n, kk):
    """The float engine's gate beside its up: the bits of the stacked product and the activation's own launch, from fewer
    values of k than a stage holds to more than all stages do, with both numbers of stages."""
    k = kernels(torch.float32)
    a, w = rnd((m, kk), torch.float32, 70), rnd((2 * n, kk), torch.float32, 71, 0.3)
    both, want = torch.empty((m, 2 * n), device="cuda"), torch.empty((m, n), device="cuda")
    k.gemm(a, w, both)
    k.silu_mul(both, want)
    shifted = torch.empty(m * kk + 1, device="cuda")[1:].view(m, kk).copy_(a)      # rows 4 bytes off
    assert k.gated_strips(m, n, kk) and not k.gated_strips(1024, 4096, 64)
    for rows in (a, shifted):
        out = torch.full((m, n), float("nan"), device="cuda")
        k.gemm_gated_silu(rows, w, out)
        assert torch.equal(out, want)


@pytest.mark.parametrize("rows,width", [(3, 5), (8, 1024), (2, 1023), (5, 1025), (4, 5120), (2, 5121), (1, 8200)])
def test_add_rmsnorm_float_widths(rows, width):
    """The float engine's norm at widths around those whose rows stay in registers, with the residual written back and without:
    a thread adds the squares of every 256th value in ascending order."""
    k = kernels(torch.float32)
    h, delta, w = rnd((rows, width), torch.float32, 72), rnd((rows, width), torch.float32, 73), rnd((width,), torch.float32, 74)
    want_h = torch.addcmul(h, delta, torch.ones_like(delta))
    squares = torch.nn.functional.pad(want_h, (0, -width % 256)).view(rows, -1, 256).double()
    total = torch.zeros((rows, 256), dtype=torch.float64, device="cuda")
    for i in range(squares.shape[1]):
        total = (total + squares[:, i] * squares[:, i]).float().double()      # (fmaf: one rounding of a sum that 64 bits hold nearly exactly)
    mean = total.sum(1) / width
    for write in (True, False):
        x, out = h.clone(), torch.full((rows, width), float("nan"), device="cuda")
        k.add_rmsnorm(x, delta, w, out, 1e-6, write_h=write)
        assert torch.equal(x, want_h if write else h)
        # 256 partial sums are added in 32 bits over nine levels; then a division, a square root, a division and two products
        assert bool(((out.double() - want_h.double() * torch.rsqrt(mean + 1e-6)[:, None] * w.double()).abs()
                     <= 16 * 2.0 ** -24 * out.double().abs() + 1e-30).all())


@pytest.mark.parametrize("shape", [0, 1, 2, 3])
@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("mnk", [(65, 70, 64), (300, 257, 192), (513, 1000, 128), (128, 256, 1024), (1, 5, 320)])
def test_gemm_wide_every_shape(shape, gated, mnk):
    """The many-row kernel in each of its workgroup shapes, plain and with the feed-forward's activation
    in its epilogue, at sizes that fill no tile; and the same bits from every shape (an output element is
    one chain of matrix-core sums over k, whatever tile it lies in)."""
    from mini_llm_runtime_amd.kernels.ops import _c_int, _p, _stream
    m, n, kk = mnk
    lib = kernels(torch.bfloat16)._lib("gemm")
    a = rnd((m, kk), torch.bfloat16, 60)
    w = rnd((2 * n if gated else n, kk), torch.bfloat16, 61, 0.3)

    def run(which, out_dtype):
        out = torch.full((m, n), float("nan"), dtype=out_dtype, device="cuda")
        rc = lib.mlr_gemm_wide(_p(a), _p(w), _p(out), _c_int(m), _c_int(n), _c_int(kk),
                               _c_int(1 if out_dtype == torch.float32 else 0), _c_int(which), _c_int(1 if gated else 0),
                               _stream())
        assert rc == 0, rc
        return out
    out = run(shape, torch.bfloat16)
    if gated:
        g = a.double() @ w.double()[:n].T
        u = a.double() @ w.double()[n:].T
        want = g / (1 + torch.exp(-g)) * u
    else:
        want = a.double() @ w.double().T
        torch.testing.assert_close(run(shape, torch.float32).double(), want, atol=1e-4 * math.sqrt(kk), rtol=1e-5)
    torch.testing.assert_close(out.double(), want, atol=2e-2 * float(want.abs().max()), rtol=2e-2)
    assert torch.equal(out, run(0, torch.bfloat16))
    assert torch.equal(out, run(-1, torch.bfloat16))


@pytest.mark.parametrize("mnk", [(17, 40, 64), (31, 257, 1216), (32, 1041, 1280), (33, 96, 1344), (48, 704, 1024), (63, 1127, 2048), (64, 1152, 2816), (32, 2050, 4032), (29, 520, 576)])
def test_gemm_few_rows_narrow_tiles(mnk):
    """17 to 64 rows on the tiles made for them, from fewer blocks of k than the LDS holds (20 at most) to several rounds of it, in
    whole pairs and not, with parts of k that end within a pair: the bits of the few-row kernel from each of them, from the entry points
    that choose among them, and with an activation; no gated form of strips of 16 columns, none beyond 64 rows."""
    from mini_llm_runtime_amd.kernels.ops import _c_int, _p, _stream
    m, n, kk = mnk
    k = kernels(torch.bfloat16)
    lib = k._lib("gemm")
    a = rnd((m, kk), torch.bfloat16, 68)
    w = rnd((2 * n, kk), torch.bfloat16, 69, 0.3)

    def run(shape, gated=0, rows=m):
        out = torch.full((m, n if gated else 2 * n), float("nan"), dtype=torch.bfloat16, device="cuda")
        rc = lib.mlr_gemm_wide(_p(a), _p(w), _p(out), _c_int(rows), _c_int(out.shape[1]), _c_int(kk), _c_int(0), _c_int(shape), _c_int(gated), _stream())
        assert rc == (-1 if rows > 64 or gated and shape in (10, 12) else 0)
        return out
    product, silu = torch.empty((m, 2 * n), dtype=torch.bfloat16, device="cuda"), torch.empty((m, n), dtype=torch.bfloat16, device="cuda")
    assert lib.mlr_gemm(_p(a), _p(w), _p(product), _c_int(m), _c_int(2 * n), _c_int(kk), _c_int(0), _stream()) == 0
    assert lib.mlr_gemm_gated_silu(_p(a), _p(w), _p(silu), _c_int(m), _c_int(n), _c_int(kk), _stream()) == 0
    want = a.double() @ w.double().T
    # (kk roundings of 2^-24 of the sum of the sizes, and bfloat16's 2^-9)
    assert bool(((product.double() - want).abs() <= kk * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 2.0 ** -8 * want.abs()).all())
    for shape in (10, 11, 12, 13, 14, 15, 16, -2):
        assert torch.equal(run(shape), product), shape
        assert shape in (10, 12) or torch.equal(run(shape, 1), silu), shape
    run(-2, rows=65)                                       # (refused before anything is launched)
    out, two, one = torch.empty_like(product), torch.empty_like(silu), torch.empty_like(silu)
    if kk <= 2816:
        k.gemm(a, w, out, library=False)
        assert torch.equal(out, product)
        k.gemm_gated_silu(a, w, two)
        assert torch.equal(two, silu)
    k.silu_mul(product, two)
    k.gemm_activated(a, w, one, "silu")
    assert torch.equal(one, two)


@pytest.mark.parametrize("mnk", [(1, 8, 64), (65, 36, 128), (97, 193, 320), (257, 385, 448), (300, 1001, 832), (513, 520, 1024)])
def test_gemm_wide_tiles_and_epilogues(mnk):
    """Every tile of the many-row kernel at sizes around its edges, from fewer blocks of k than the LDS holds to several
    rounds of it: the plain product within the rounding of its 32-bit sums and of bfloat16, the same bits from every tile,
    and every activation in the epilogue with the bits of the product and the activation's own launch."""
    from mini_llm_runtime_amd.kernels.ops import _c_int, _p, _stream
    m, n, kk = mnk
    k = kernels(torch.bfloat16)
    lib = k._lib("gemm")
    a = rnd((m, kk), torch.bfloat16, 66)
    w = rnd((2 * n, kk), torch.bfloat16, 67, 0.3)

    def run(shape, gated=0):
        out = torch.full((m, n if gated else 2 * n), float("nan"), dtype=torch.bfloat16, device="cuda")
        assert lib.mlr_gemm_wide(_p(a), _p(w), _p(out), _c_int(m), _c_int(out.shape[1]), _c_int(kk), _c_int(0), _c_int(shape), _c_int(gated), _stream()) == 0
        return out
    product, silu = run(-1), run(-1, 1)
    chain = product
    want = a.double() @ w.double().T
    # a sum of kk products in 32 bits is off by at most kk roundings of 2^-24 of the sum of their sizes; bfloat16 adds 2^-9
    bound = kk * 2.0 ** -24 * (a.double().abs() @ w.double().abs().T) + 2.0 ** -8 * want.abs()
    assert bool(((product.double() - want).abs() <= bound).all())
    for shape in range(10):
        assert torch.equal(run(shape), chain) and torch.equal(run(shape, 1), silu), shape
    if m <= 64:
        product = run(-2)                                  # (the activations' products are then those of few rows)
    two, one = torch.empty((m, n), dtype=torch.bfloat16, device="cuda"), torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    for kind in ("silu", "gelu_tanh", "relu", "clamped"):
        if kind == "silu":
            k.silu_mul(product, two)
        elif kind == "clamped":
            k.clamped_glu(product, two, 0.7, 1.702)
        else:
            k.gated_act_mul(product, two, kind)
        k.gemm_activated(a, w, one, kind, 0.7, 1.702)
        assert torch.equal(one, two), kind
    for kind in ("relu_squared", "gelu_erf"):
        whole = torch.empty_like(product)
        k.plain_act(product, whole, kind)
        got = torch.full_like(product, float("nan"))
        k.gemm_activated(a, w, got, kind)
        assert torch.equal(got, whole), kind
    shifted = torch.empty(m * kk + 1, dtype=torch.bfloat16, device="cuda")[1:].view(m, kk).copy_(a)      # rows 2 bytes off
    k.gemm_activated(shifted, w, one, "relu")
    k.gated_act_mul(product, two, "relu")
    assert torch.equal(one, two)
    out = torch.full((m, 2 * n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm(shifted, w, out)
    assert bool(((out.double() - want).abs() <= bound).all())


@pytest.mark.parametrize("m,n,kk", [(65, 8072, 8192), (67, 16000, 64), (75, 111800, 1984), (99, 80000, 8128), (130, 4040, 4032), (333, 1576, 8000),
                                    (333, 25000, 8192), (509, 32800, 2048), (701, 760, 7360), (997, 536, 3328), (1001, 8376, 8704), (70, 34944, 8704), (1499, 11100, 1088),
                                    (2047, 264, 2048), (2001, 4192, 8192), (2049, 8184, 2048), (4099, 2040, 5056), (8191, 1016, 8192), (8190, 2040, 1920)])
def test_the_library_adds_alike_where_models_with_a_router_leave_it(m, n, kk):
    """Products inside and at the edges of `library_adds_alike`: the vendor library's own first choice has the many-row kernel's bits,
    alone and with the activation behind it in a launch of its own.  (Row counts that the library does not time.)"""
    from mini_llm_runtime_amd.kernels.ops import _c_int, _p, _stream
    k = kernels(torch.bfloat16)
    assert k.library_adds_alike(m * n, kk) and m % 64 != 0
    a = rnd((m, kk), torch.bfloat16, 98)
    w = torch.empty((n, kk), dtype=torch.bfloat16, device="cuda").normal_(generator=torch.Generator("cuda").manual_seed(99)).mul_(0.05)
    out, own = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    k.wide_product = lambda *sizes: False
    k.gemm(a, w, out)
    assert k._lib("gemm").mlr_gemm_wide(_p(a), _p(w), _p(own), _c_int(m), _c_int(n), _c_int(kk), _c_int(0), _c_int(-1), _c_int(0), _stream()) == 0
    assert torch.equal(out, own)
    act, one = (torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    k.silu_mul(out, act)
    k.gemm_activated(a, w, one, "silu")
    assert torch.equal(act, one)


@pytest.mark.parametrize("m,n,kk", [(33, 5632, 1408), (33, 5632, 4096), (47, 5640, 2048), (48, 8192, 2048), (63, 16384, 4096), (50, 11264, 1088), (17, 8448, 2112),
                                    (25, 8456, 4096), (32, 16384, 3072)])
def test_up_to_64_rows_add_as_the_library_does_in_a_model_with_a_router(m, n, kk):
    """Inside and at the edges of `library_adds_few_alike`: the library's bits, plain and with the activation behind it."""
    from mini_llm_runtime_amd.kernels import Kernels
    k, library = Kernels(torch.bfloat16, routed=True), Kernels(torch.bfloat16, routed=True)
    assert k.wide_product(m, n, kk) and k.wide_product(m, n // 2, kk, "silu") and k.one_sum(m, kk)
    library.wide_product = lambda *sizes: False
    a, w = rnd((m, kk), torch.bfloat16, 41), rnd((n, kk), torch.bfloat16, 42, 0.05)
    out, own = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    library.gemm(a, w, out)
    k.gemm(a, w, own)
    assert torch.equal(out, own)
    act, one = (torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    for kind in ("silu", "relu", "clamped"):
        k._product_then_activation(a, w, act, kind, 7.0, 1.702)
        k.gemm_activated(a, w, one, kind, 7.0, 1.702)
        assert torch.equal(act, one), kind


@pytest.mark.parametrize("m,n,kk", [(17, 6144, 2048), (32, 2816, 2048), (33, 512, 1024), (64, 12288, 1024), (24, 8448, 1984), (48, 30, 704)])
def test_the_narrow_tiles_of_a_model_with_a_router_have_the_streamed_kernels_bits(m, n, kk):
    from mini_llm_runtime_amd.kernels import Kernels
    k, streamed = Kernels(torch.bfloat16, routed=True), Kernels(torch.bfloat16, routed=True)
    assert k.few_product(m, n, kk) and not k.wide_product(m, n, kk)
    streamed.few_product = lambda *sizes: False
    a, w = rnd((m, kk), torch.bfloat16, 43), rnd((n, kk), torch.bfloat16, 44, 0.05)
    out, own = (torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    streamed.gemm(a, w, out)
    k.gemm(a, w, own)
    assert torch.equal(out, own)
    act, one = (torch.full((m, n // 2), float("nan"), dtype=torch.bfloat16, device="cuda") for _ in range(2))
    streamed.gemm_gated_silu(a, w, act)
    k.gemm_gated_silu(a, w, one)
    assert torch.equal(act, one)


def test_gemm_float_of_an_inner_size_beyond_32_bits_of_bytes():
    """16 rows of 2^26 floats are 2^32 bytes, one more than the few-row kernel's loads reach: the product is the tiles', plain and
    beside an activation.  (Whole numbers: exact.)"""
    k, kk = kernels(torch.float32), 1 << 26
    a, w = torch.zeros((1, kk), device="cuda"), torch.full((2, kk), 3.0, device="cuda")
    a[0, ::1 << 22] = 1
    a[0, -1] = 2
    out, act = torch.full((1, 2), float("nan"), device="cuda"), torch.full((1, 1), float("nan"), device="cuda")
    k.gemm(a, w, out)
    assert out.tolist() == [[54.0, 54.0]]
    assert not k.gated_strips(1, 1, kk)
    k.silu_mul(out, act)
    assert abs(act.item() - 54.0 * 54.0) < 1e-3


@pytest.mark.parametrize("dtype,m,n,kk", [(torch.bfloat16, 100, 3000, 512), (torch.bfloat16, 20, 3000, 512), (torch.float32, 8, 1000, 2048)])
def test_activations_behind_a_weight_off_16_bytes(dtype, m, n, kk):
    """A weight that is a view off 16 bytes is read where it lies: no call copies it, and the feed-forward's choice of a way looks at
    it.  The results are the product's and the activation's own launches."""
    k = kernels(dtype)
    a, aligned = rnd((m, kk), dtype, 96), rnd((2 * n, kk), dtype, 97, 0.3)
    w = torch.empty(2 * n * kk + 1, dtype=dtype, device="cuda")[1:].view(2 * n, kk).copy_(aligned)
    one, want, both = (torch.empty((m, c), dtype=dtype, device="cuda") for c in (n, n, 2 * n))
    k.gemm(a, w, both)
    k.silu_mul(both, want)
    calls = [lambda: k.gemm_gated_silu(a, w, one)] if m > 64 or dtype == torch.float32 else []
    if dtype == torch.bfloat16:
        calls.append(lambda: k.gemm_activated(a, w, one, "silu"))
        assert not k.wide_product(m, n, kk, "silu", w) and k.gated_silu_fused(m, kk, w) == (m <= 64)
    assert not k.gated_strips(m, n, kk, w)
    for call in calls:
        one.fill_(float("nan"))
        torch.cuda.synchronize()
        torch.cuda.reset_peak_memory_stats()
        before = torch.cuda.memory_allocated()
        call()
        assert torch.equal(one, want)
        assert torch.cuda.max_memory_allocated() - before < w.numel() * w.element_size()
    if dtype == torch.bfloat16:
        whole, got = both.clone(), torch.full_like(both, float("nan"))
        k.plain_act(whole, whole, "gelu_erf")
        k.gemm_activated(a, w, got, "gelu_erf")
        assert torch.equal(got, whole)


def test_gemm_wide_rows_do_not_depend_on_the_batch():
    """More than 64 rows with an inner size that is a multiple of 64: the tile shape follows the number of
    rows, a row's bits do not."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16, library_gemm=False)
    a = rnd((700, 256), torch.bfloat16, 62)
    w = rnd((1100, 256), torch.bfloat16, 63)

    def run(lo, hi):
        out = torch.empty((hi - lo, 1100), dtype=torch.bfloat16, device="cuda")
        k.gemm(a[lo:hi].contiguous(), w, out)
        return out
    full = run(0, 700)
    for lo, hi in [(0, 65), (100, 400), (630, 700), (1, 699)]:
        assert torch.equal(run(lo, hi), full[lo:hi])


def test_gemm_gated_silu_many_rows():
    """Without the library the feed-forward's first projection keeps its fused activation at any number
    of rows (inner size a multiple of 64)."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.bfloat16, library_gemm=False)
    assert k.gated_silu_fused(2048, 1024) and not k.gated_silu_fused(2048, 1000)
    # beside the library it stays the way while the inner size is short
    assert kernels(torch.bfloat16).gated_silu_fused(2048, 1024) and kernels(torch.bfloat16).gated_silu_fused(256, 2048)
    assert not kernels(torch.bfloat16).gated_silu_fused(2048, 4096) and not kernels(torch.bfloat16).gated_silu_fused(512, 2048)
    m, n, kk = 333, 424, 384
    a = rnd((m, kk), torch.bfloat16, 64)
    w = rnd((2 * n, kk), torch.bfloat16, 65, 0.3)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_gated_silu(a, w, out)
    g = a.double() @ w.double()[:n].T
    u = a.double() @ w.double()[n:].T
    want = g / (1 + torch.exp(-g)) * u
    torch.testing.assert_close(out.double(), want, atol=2e-2 * float(want.abs().max()), rtol=2e-2)


def plain_rope(x, pos, base):
    """x [T, H, D] float64 by the plain implementation's rotation (angles held in 32-bit, as the
    reference computes them)."""
    from plain.qwen3_plain import rope_cos_sin, rope_rotate
    cos, sin = rope_cos_sin(pos.numpy(), x.shape[-1], base)
    return torch.from_numpy(rope_rotate(x.numpy(), cos, sin))


def rope_table(max_pos, dim, base):
    from mini_llm_runtime_amd.config import PositionSpec
    from mini_llm_runtime_amd.parts.rope import RopeSplitHalf
    return RopeSplitHalf(PositionSpec("rope_split_half", dim, base)).rotation_table(max_pos, "cuda")


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(1, 1, 16, 4), (8, 2, 128, 16), (6, 3, 48, 8), (16, 16, 256, 32), (5, 1, 32, 1)])
def test_qk_norm_rope_kv(dtype, shape):
    """Positions around page edges and far ones (tests/cuda_ops_tests.cu:326); shuffled pages."""
    hq, hkv, d, page = shape
    k = kernels(dtype)
    positions = [0, 1, page - 1, page, page + 1, 2 * page + 3, 1535, 2047]
    positions = sorted(set(p for p in positions))
    m = len(positions)
    max_blocks = 2048 // page + 1
    # two slots: even rows in slot 1, odd rows in slot 0; pages handed out in a shuffled order
    slots = torch.tensor([1 - (i % 2) for i in range(m)], dtype=torch.int32)
    n_pages = 2 * m + 3
    perm = torch.randperm(n_pages, generator=torch.Generator().manual_seed(11)).tolist()
    table = torch.full((2, max_blocks), -1, dtype=torch.int32)
    for i, p in enumerate(positions):
        table[slots[i], p // page] = perm.pop()
    qkv = rnd((m, (hq + 2 * hkv) * d), dtype, 12)
    qw, kw = rnd((d,), torch.float32, 13) + 1, rnd((d,), torch.float32, 14) + 1
    eps, base = 1e-5, 1e6
    rope = rope_table(2048, d, base)
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype, device="cuda")
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype, device="cuda")
    q_out = torch.empty((m, hq * d), dtype=dtype, device="cuda")
    pos_t = torch.tensor(positions, dtype=torch.int32)
    k.qk_norm_rope_kv(qkv, q_out, k_pages, v_pages, table.cuda(), slots.cuda(), pos_t.cuda(), qw, kw, eps,
                      rope, hq, hkv, d, page)
    x = qkv.double().cpu()
    q = x[:, :hq * d].view(m, hq, d)
    kk = x[:, hq * d:(hq + hkv) * d].view(m, hkv, d)
    v = x[:, (hq + hkv) * d:].view(m, hkv, d)

    def norm(t, w):
        return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + eps) * w.double().cpu()
    q_want = plain_rope(norm(q, qw), pos_t, base)
    k_want = plain_rope(norm(kk, kw), pos_t, base)
    torch.testing.assert_close(q_out.double().cpu().view(m, hq, d), q_want, **tol(dtype))
    written = torch.zeros((n_pages, page), dtype=torch.bool)
    for i, p in enumerate(positions):
        pg = table[slots[i], p // page].item()
        written[pg, p % page] = True
        torch.testing.assert_close(k_pages[pg, :, p % page].double().cpu(), k_want[i], **tol(dtype))
        assert torch.equal(v_pages[pg, :, :, p % page].cpu(), qkv[i, (hq + hkv) * d:].view(hkv, d).cpu())
    # nothing else was touched
    untouched = ~written[:, None, :, None].expand(n_pages, hkv, page, d)
    assert torch.isnan(k_pages.float().cpu()[untouched]).all()
    assert torch.isnan(v_pages.float().cpu().transpose(2, 3)[untouched]).all()
    # no norm, no rotation, no cache write
    k2 = torch.full_like(k_pages, float("nan"))
    k.qk_norm_rope_kv(qkv, q_out, k2, v_pages, table.cuda(), slots.cuda(), pos_t.cuda(), None, None, 0.0,
                      None, hq, hkv, d, page, write_cache=False)
    assert torch.equal(q_out.cpu(), qkv[:, :hq * d].cpu())
    assert torch.isnan(k2.float()).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", [
    # (q heads, kv heads, head_dim, channels turned, interleaved, rows)
    (4, 2, 16, 8, True, 5), (4, 2, 16, 16, True, 70), (2, 1, 64, 32, False, 9), (2, 1, 64, 32, False, 130),
    (3, 3, 48, 2, True, 4), (2, 2, 128, 64, True, 66), (1, 1, 20, 10, False, 3), (2, 1, 256, 128, False, 2)])
def test_rotation_of_part_of_a_head_in_either_pairing(dtype, case):
    """The rotation kernel takes the extent and the pairing from its caller: the first `turned` channels of a
    head in pairs (j, j + turned / 2) or (2 j, 2 j + 1), the rest unrotated; the per-head norm spans the whole
    head either way.  (70 and 130 rows: the vector kernel for many rows must not be taken for these.)"""
    hq, hkv, d, turned, interleaved, rows = case
    k = kernels(dtype)
    page, eps = 16, 1e-5
    width = (hq + 2 * hkv) * d
    qkv = rnd((rows, width), dtype, 300)
    qw, kw = rnd((d,), torch.float32, 301) + 1, rnd((d,), torch.float32, 302) + 1
    n_pages = (rows + page - 1) // page + 1
    table = torch.arange(n_pages, dtype=torch.int32).flip(0).view(1, -1).contiguous().cuda()
    slots = torch.zeros(rows, dtype=torch.int32, device="cuda")
    pos = torch.arange(rows, dtype=torch.int32, device="cuda")
    angle = torch.arange(rows, dtype=torch.float64)[:, None] * (100.0 ** (-2.0 * torch.arange(turned // 2, dtype=torch.float64) / turned))[None, :]
    rope = torch.cat([torch.cos(angle), torch.sin(angle)], dim=1).float().cuda()
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype, device="cuda")
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype, device="cuda")
    q_out = torch.full((rows, hq * d), float("nan"), dtype=dtype, device="cuda")
    k.qk_norm_rope_kv(qkv, q_out, k_pages, v_pages, table, slots, pos, qw, kw, eps, rope, hq, hkv, d, page,
                      interleaved=interleaved)

    def want(x, w):                                      # x [rows, heads, d] float64
        x = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + eps) * w.double().cpu()
        c, s = torch.cos(angle)[:, None, :], torch.sin(angle)[:, None, :]
        out = x.clone()
        if interleaved:
            a, b = x[..., 0:turned:2], x[..., 1:turned:2]
            out[..., 0:turned:2], out[..., 1:turned:2] = a * c - b * s, a * s + b * c
        else:
            a, b = x[..., :turned // 2], x[..., turned // 2:turned]
            out[..., :turned // 2], out[..., turned // 2:turned] = a * c - b * s, a * s + b * c
        return out
    x = qkv.double().cpu()
    torch.testing.assert_close(q_out.double().cpu().view(rows, hq, d), want(x[:, :hq * d].view(rows, hq, d), qw), **tol(dtype))
    k_want = want(x[:, hq * d:(hq + hkv) * d].view(rows, hkv, d), kw)
    for r in range(rows):
        pg = int(table[0, r // page])
        torch.testing.assert_close(k_pages[pg, :, r % page].double().cpu(), k_want[r], **tol(dtype))
        assert torch.equal(v_pages[pg, :, :, r % page].cpu(), qkv[r, (hq + hkv) * d:].view(hkv, d).cpu())


def plain_attention(q, keys, values, scale, window):
    """One query row over its visible keys, float64.  q [Hq, D]; keys, values [L, Hkv, D]."""
    hq, hkv = q.shape[0], keys.shape[1]
    g = hq // hkv
    L = keys.shape[0]
    lo = 0 if window is None else max(0, L - window)
    out = torch.zeros_like(q)
    for h in range(hq):
        s = (keys[lo:, h // g] @ q[h]) * scale
        a = torch.softmax(s, dim=0)
        out[h] = a @ values[lo:, h // g]
    return out


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("case", [
    # (q heads, kv heads, head_dim, page, lengths of the requests, window, split_keys)
    (4, 1, 16, 16, [1, 17, 33], None, 0),
    (4, 2, 128, 16, [15, 16, 17, 127, 128, 129], None, 0),
    (16, 8, 128, 16, [300, 1], None, 64),
    (6, 3, 48, 8, [70, 131], None, 64),
    (20, 1, 32, 32, [100], None, 0),
    (4, 4, 256, 16, [65], None, 0),
    (4, 2, 64, 16, [200, 40], 33, 0),
    (4, 2, 64, 16, [200, 40], 64, 128),
    (2, 1, 16, 4, [1000], None, 256),
    (6, 3, 48, 32, [100, 70], None, 0),
    (32, 2, 64, 16, [130, 5], None, 64),
    (8, 8, 80, 16, [77], 40, 0),
    (16, 8, 128, 16, [530, 3], None, 0),
    (4, 1, 96, 32, [150], 50, 0),
    (14, 2, 192, 16, [40], None, 0),
    (2, 1, 224, 16, [40], None, 0),
    (4, 2, 32, 16, [300], 70, 0),
    (8, 2, 64, 64, [333, 20], None, 128),
    (4, 2, 128, 128, [400, 130], None, 0),
    (6, 2, 96, 256, [300], 100, 64),
    (3, 1, 112, 32, [200], None, 0),
    (10, 2, 16, 16, [150, 64], 64, 0),
])
def test_paged_attention(dtype, case):
    """Every length is one request whose LAST token is the query (a decoded token) plus, for the
    first request, a query at every position (a whole prompt); pages shuffled.  Shapes after
    tests/cuda_layer_tests.cpp:528-536."""
    hq, hkv, d, page, lengths, window, split_keys = case
    k = kernels(dtype)
    g = torch.Generator().manual_seed(20)
    max_len = max(lengths)
    max_blocks = (max_len + page - 1) // page
    n_pages = sum((L + page - 1) // page for L in lengths) + 2
    perm = torch.randperm(n_pages, generator=g).tolist()
    table = torch.full((len(lengths), max_blocks), -1, dtype=torch.int32)
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype)
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype)
    keys, values = [], []
    for s, L in enumerate(lengths):
        kk = torch.randn((L, hkv, d), generator=g).to(dtype)
        vv = torch.randn((L, hkv, d), generator=g).to(dtype)
        keys.append(kk)
        values.append(vv)
        for b in range((L + page - 1) // page):
            pg = perm.pop()
            table[s, b] = pg
            n = min(page, L - b * page)
            k_pages[pg, :, :n] = kk[b * page:b * page + n].transpose(0, 1)
            v_pages[pg, :, :, :n] = vv[b * page:b * page + n].permute(1, 2, 0)
    rows = [(0, p) for p in range(lengths[0])] + [(s, L - 1) for s, L in enumerate(lengths) if s > 0]
    m = len(rows)
    q = (torch.randn((m, hq, d), generator=g) * 2).to(dtype)
    scale = 1 / math.sqrt(d)
    out = torch.full((m, hq * d), float("nan"), dtype=dtype, device="cuda")
    slots = torch.tensor([r[0] for r in rows], dtype=torch.int32).cuda()
    pos = torch.tensor([r[1] for r in rows], dtype=torch.int32).cuda()
    max_splits, partial = 1, None
    if split_keys:
        max_splits = (max_len + split_keys - 1) // split_keys
        partial = torch.full((k.attention_partial_numel(m, hq, d, max_splits),), float("nan"), device="cuda")
    k.paged_attention(q.view(m, hq * d).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), slots, pos, out,
                      hq, hkv, d, page, scale, window=window, split_keys=split_keys, max_splits=max_splits,
                      partial=partial)
    got = out.double().cpu().view(m, hq, d)
    wants = [plain_attention(q[i].double(), keys[s][:p + 1].double(), values[s][:p + 1].double(), scale, window)
             for i, (s, p) in enumerate(rows)]
    for i in range(m):
        torch.testing.assert_close(got[i], wants[i], **tol(dtype))
    if not k.mfma_attention_supported(hq, hkv, d, page):
        return
    # the matrix-core kernel: the first request's rows in groups of consecutive tokens, the others alone
    tq = max(1, 16 // (hq // hkv))
    first = list(range(0, lengths[0], tq)) + list(range(lengths[0], m))
    count = [min(tq, lengths[0] - r) for r in range(0, lengths[0], tq)] + [1] * (m - lengths[0])
    out2 = torch.full((m, hq * d), float("nan"), dtype=dtype, device="cuda")
    if partial is not None:
        partial.fill_(float("nan"))
    k.attention_mfma(q.view(m, hq * d).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), slots, pos, out2,
                     torch.tensor(first, dtype=torch.int32).cuda(), torch.tensor(count, dtype=torch.int32).cuda(),
                     len(first), hq, hkv, d, page, scale, window=window, split_keys=split_keys,
                     max_splits=max_splits, partial=partial)
    got = out2.double().cpu().view(m, hq, d)
    for i in range(m):
        torch.testing.assert_close(got[i], wants[i], **tol(dtype))
    if not k.prefill_attention_supported(hq, hkv, d, page):
        return
    # the kernel for prompt portions: the first request's rows in groups of up to 4 tq tokens; other rows untouched
    big = 4 * tq
    first = list(range(0, lengths[0], big))
    count = [min(big, lengths[0] - r) for r in first]
    out3 = torch.full((m, hq * d), float("nan"), dtype=dtype, device="cuda")
    k.attention_prefill(q.view(m, hq * d).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), slots, pos, out3,
                        torch.tensor(first, dtype=torch.int32).cuda(), torch.tensor(count, dtype=torch.int32).cuda(),
                        len(first), hq, hkv, d, page, scale, window=window)
    got = out3.double().cpu().view(m, hq, d)
    for i in range(lengths[0]):
        torch.testing.assert_close(got[i], wants[i], **tol(dtype))
    assert torch.isnan(out3[lengths[0]:].float()).all()
    if not k.tiles_attention_supported(hq, hkv, d, page):
        return
    # the 32x32-tile kernel for prompt portions, with both sizes of workgroup: groups of as many tokens as a
    # workgroup takes, and of fewer
    # (workgroups of 128 columns that take two groups each, and one: small batches would only meet the latter)
    for columns, big, split, pairing in ((128, k.tiles_group_tokens(hq, hkv, 128), 0, "pairs"), (128, 8 * tq, 0, "pairs"),
                                         (128, 8 * tq, 0, "single"),
                                         (64, k.tiles_group_tokens(hq, hkv, 64), 0, "auto"), (64, 3 * tq, 0, "auto"),
                                         (128, k.tiles_group_tokens(hq, hkv, 128), 64, "auto"), (64, 3 * tq, 128, "auto")):
        first = list(range(0, lengths[0], big))
        count = [min(big, lengths[0] - r) for r in first]
        out4 = torch.full((m, hq * d), float("nan"), dtype=dtype, device="cuda")
        splits, part = 1, None
        if split:
            splits = (max_len + split - 1) // split
            part = torch.full((k.attention_partial_numel(m, hq, d, splits),), float("nan"), device="cuda")
        k.attention_tiles(q.view(m, hq * d).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), slots, pos, out4,
                          torch.tensor(first, dtype=torch.int32).cuda(), torch.tensor(count, dtype=torch.int32).cuda(),
                          len(first), hq, hkv, d, page, scale, window=window, columns=columns,
                          split_keys=split, max_splits=splits, partial=part, pairing=pairing)
        got = out4.double().cpu().view(m, hq, d)
        for i in range(lengths[0]):
            torch.testing.assert_close(got[i], wants[i], **tol(dtype))
        assert torch.isnan(out4[lengths[0]:].float()).all()


@pytest.mark.parametrize("hq,hkv,page,before,n,window,split", [
    (2, 1, 16, 0, 1, None, 0), (16, 8, 16, 0, 300, None, 0), (16, 8, 16, 63, 65, None, 0), (8, 1, 16, 255, 130, None, 0),
    (4, 4, 32, 320, 193, None, 0), (4, 2, 64, 511, 129, None, 0), (4, 2, 256, 700, 200, None, 0), (16, 1, 128, 449, 33, None, 0),
    (4, 2, 16, 500, 150, 200, 0), (4, 2, 64, 600, 97, 70, 0), (4, 2, 16, 900, 70, None, 256), (2, 1, 32, 1000, 64, 500, 128)])
def test_prompt_portions_of_head_size_128(hq, hkv, page, before, n, window, split):
    """The prompt portions' kernel whose blocks go to LDS past the registers, at portions that start and end beside the edges
    of blocks and pages, with pages smaller and larger than a block, behind a window whose pages were given back, in key
    ranges; keys not written yet hold NaN, and so does every page that is not the request's.  The same bits every time."""
    k = kernels(torch.bfloat16)
    d, ctx, scale = 128, before + n, 128 ** -0.5
    blocks = (ctx + page - 1) // page
    keys, values = rnd((ctx, hkv, d), torch.bfloat16, 90), rnd((ctx, hkv, d), torch.bfloat16, 91)
    q = rnd((n, hq * d), torch.bfloat16, 92, 2.0)
    ids = torch.randperm(blocks + 2, generator=torch.Generator().manual_seed(93))[:blocks].cuda()
    k_pages = torch.full((blocks + 2, hkv, page, d), float("nan"), dtype=torch.bfloat16, device="cuda")
    v_pages = torch.full((blocks + 2, hkv, d, page), float("nan"), dtype=torch.bfloat16, device="cuda")
    at = torch.arange(ctx, device="cuda")
    k_pages[ids[at // page], :, at % page] = keys
    v_pages[ids[at // page], :, :, at % page] = values
    table = torch.full((1, blocks + 1), -1, dtype=torch.int32, device="cuda")
    table[0, :blocks] = ids.int()
    if window is not None:
        gone = max(0, before + 1 - window) // page
        k_pages[ids[:gone]], v_pages[ids[:gone]], table[0, :gone] = float("nan"), float("nan"), -1
    slots, pos = torch.zeros(n, dtype=torch.int32, device="cuda"), torch.arange(before, ctx, dtype=torch.int32, device="cuda")
    g = hq // hkv
    seen = at[None] <= pos[:, None]
    if window is not None:
        seen &= at[None] > pos[:, None] - window
    want, size = torch.empty((n, hq, d), dtype=torch.float64, device="cuda"), torch.empty((n, hq, d), dtype=torch.float64, device="cuda")
    for head in range(hq):
        w = torch.softmax((q.view(n, hq, d)[:, head].double() @ keys[:, head // g].double().T * scale).masked_fill(~seen, -math.inf), -1)
        want[:, head], size[:, head] = w @ values[:, head // g].double(), w @ values[:, head // g].double().abs()
    # a probability is rounded to bfloat16 (2^-9 of itself, in numerator and denominator) and its score is a 32-bit sum; so is the result
    bound = (2.0 ** -8 + 1e-4) * size + 2.0 ** -8 * want.abs()
    widths = []
    for columns in (128, 64):
        for cap in {columns // g, max(1, columns // g - 3)}:
            first = list(range(0, n, cap))
            splits = -(-ctx // split) if split else 1
            part = torch.full((k.attention_partial_numel(n, hq, d, splits),), float("nan"), device="cuda") if split else None
            before_out = None
            for _ in range(3):
                out = torch.full((n, hq * d), float("nan"), dtype=torch.bfloat16, device="cuda")
                k.attention_tiles(q, k_pages, v_pages, table, slots, pos, out, torch.tensor(first, dtype=torch.int32, device="cuda"),
                                  torch.tensor([min(cap, n - r) for r in first], dtype=torch.int32, device="cuda"), len(first), hq, hkv, d, page,
                                  scale, window=window, columns=columns, split_keys=split, max_splits=splits, partial=part)
                assert bool(((out.double().view(n, hq, d) - want).abs() <= bound).all()), (columns, cap)
                assert before_out is None or torch.equal(out, before_out), (columns, cap)
                before_out = out
        widths.append(before_out.double().view(n, hq, d))
    # the two widths round the same probabilities beside other references, each by at most 2^-9 of itself, and the sums of
    # their roundings; the results to bfloat16
    assert bool(((widths[0] - widths[1]).abs() <= (2.0 ** -7 + 2e-4) * size + 2.0 ** -8 * widths[0].abs()).all())
    # over all results the two errors are about as large: one width is no less exact than the other
    errors = [float((w - want).norm() / want.norm()) for w in widths]
    assert max(errors) <= 1.1 * min(errors), errors


@pytest.mark.parametrize("d,columns", [(128, 64), (128, 128), (64, 64), (64, 128)])
def test_prompt_portions_columns_do_not_depend_on_their_neighbours(d, columns):
    """A column's reference is raised by its own probabilities alone: where one of its two lanes' sums over a tile exceeds 2^20.  The first
    block sets the reference, the second holds probabilities of some 2^16 times that: with lanes' sums just below 2^20 and of exactly 2^20
    (not raised), just above, and above in one lane of the two (raised).  With neighbours that raise theirs in the same tile and with ones
    that do not, the column's results are the same bits; and they are the softmax's, which they would not be if its lanes disagreed.
    (Scores are sums of three factors of eight bits: exact.  The probabilities of the second block lie at the edges of the rounding to
    bfloat16, each with a channel of its own, and the largest is no power of two: a raised reference shows.)"""
    k = kernels(torch.bfloat16)
    f32, scale, page, bound = np.float32, d ** -0.5, 64, 2.0 ** 20
    c2 = f32(scale) * f32(1.44269504088896340736)
    # a lane's sum is over 16 keys of a tile of 32, and over both tiles of a block where one wavefront takes them together
    tiles = 2 if d == 128 and columns == 128 else 1
    lane_of = (np.arange(32) >> (3 if d == 128 else 2)) & 1

    def lane(total):
        """Sixteen probabilities of about total / tiles of the bound together, each halfway between two bfloat16 numbers."""
        p = total * bound / tiles / 16 * (1 + (np.arange(16) - 7.5) / 32)
        ulp = 2.0 ** (np.floor(np.log2(p)) - 7)
        return (np.floor(p / ulp) + 0.5) * ulp
    # halfway, too, eight on either side of a power of two; one is put above its edge, the next below: exactly the bound
    even = (16 + np.concatenate([-np.arange(31, 74, 6) / 32, np.arange(5, 48, 6) / 16])) * (bound / 256 / tiles)
    kinds = [(lane(0.994), lane(0.994)), (even, even), (lane(1.008), lane(1.008)), (lane(1.008), lane(0.4))]
    spread = [[tiles * 2.0 ** (np.floor(np.log2(p)) - 8) for p in pair] for pair in kinds]        # whichever way an edge goes
    lows, highs = ([[tiles * p.sum() + sign * u.sum() for p, u in zip(*two)] for two in zip(kinds, spread)] for sign in (-1, 1))
    assert max(highs[0]) < bound < min(lows[2]) and lows[3][0] > bound > highs[3][1]
    assert tiles * even.sum() == bound and (even[:8] < bound / 16 / tiles).all() and (even[8:] > bound / 16 / tiles).all()
    keys, values = np.zeros((160, 4, d), f32), np.zeros((160, 4, d), f32)
    for head, lanes in enumerate(kinds):
        scores = np.zeros(128, f32)
        scores[[0, 32]] = s0 = f32(60 + head)                # (both halves of a block: either may have a reference of its own)
        for half in (64, 96):
            for side in (0, 1):
                x = ((float(f32(s0 * c2)) + np.log2(lanes[side])) / float(c2)).astype(f32)
                off = np.where(np.arange(16) % 2 == 0, 6, -6) if head == 1 else np.arange(16) % 7 - 3
                x = x + off.astype(f32) * np.spacing(x)
                scores[half + np.flatnonzero(lane_of == side)] = x
        rest = scores.copy()
        for part in range(3):                                # eight bits each
            digit = torch.tensor(rest).view(torch.int32).bitwise_and(-65536).view(torch.float32).numpy()
            keys[:128, head, part] = digit
            rest = rest - digit
        assert not rest.any()
        values[np.arange(64, 128), head, np.arange(64) % d] = 1
    k_pages = torch.tensor(keys[:128]).view(2, page, 4, d).transpose(1, 2)
    v_pages = torch.tensor(values[:128]).view(2, page, 4, d).permute(0, 2, 3, 1)
    pad = torch.zeros((1, 4, page, d))
    k_pages = torch.cat([k_pages, pad]).to(torch.bfloat16).contiguous().cuda()
    v_pages = torch.cat([v_pages, pad.transpose(2, 3)]).to(torch.bfloat16).contiguous().cuda()
    table = torch.tensor([[0, 1, 2]], dtype=torch.int32, device="cuda")
    slots, pos = torch.zeros(32, dtype=torch.int32, device="cuda"), torch.arange(128, 160, dtype=torch.int32, device="cuda")
    first, count = torch.tensor([0], dtype=torch.int32, device="cuda"), torch.tensor([32], dtype=torch.int32, device="cuda")
    got = []
    for neighbours in (0.0, 2.0):
        q = torch.zeros((32, 4, d))
        q[0, :, :3], q[1:, :, :3] = 1, neighbours
        out = torch.full((32, 4 * d), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.attention_tiles(q.view(32, -1).to(torch.bfloat16).cuda(), k_pages, v_pages, table, slots, pos, out, first, count, 1, 4, 4, d, page, scale,
                          columns=columns)
        got.append(out.view(32, 4, d))
        score = (q.double().transpose(0, 1) @ torch.tensor(keys).double().permute(1, 2, 0)) * scale               # [4, 32, 160]
        seen = torch.arange(160)[None] <= torch.arange(128, 160)[:, None]
        want = (torch.softmax(score.masked_fill(~seen, -math.inf), -1) @ torch.tensor(values).double().transpose(0, 1)).transpose(0, 1)
        # a probability is rounded to bfloat16 (2^-9 of itself, in numerator and denominator) and its score is a 32-bit sum; so is the result
        error = (out.view(32, 4, d).double().cpu() - want).abs()
        assert bool((error <= (2.0 ** -7 + 1e-4) * want).all()), (neighbours, float((error / want.clamp_min(1e-30)).max()))
    for head in range(4):
        assert bool((got[0][0, head, :64] > 0).all()) and torch.equal(got[0][0, head], got[1][0, head]), head
    # the bound lies no lower: the probabilities at it were rounded beside the first reference (a raise to their maximum would change 40
    # of the 64 results; a result at an edge of its own rounding may go either way)
    kept = even + np.where(np.arange(16) % 2 == 0, 0.5, -0.5) * 2.0 ** (np.floor(np.log2(even)) - 7)
    share = torch.zeros(64, dtype=torch.float64)
    for side in (0, 1):
        for half in (0, 32):
            share[half + np.flatnonzero(lane_of == side)] = torch.tensor(kept)
    total = share.sum() + 2 + float((63 + 1) * 2.0 ** -float(f32(f32(61) * c2)))                   # (and the other keys, with scores of zero)
    assert int((got[0][0, 1, :64].cpu() == (share / total).to(torch.bfloat16)).sum()) >= 60


@pytest.mark.parametrize("hq,hkv,d,page,window,split_keys", [(4, 2, 128, 16, None, 0), (4, 2, 128, 16, None, 64), (6, 2, 64, 32, 20, 0),
                                                             (16, 1, 48, 16, None, 0), (3, 1, 256, 16, 33, 64)])
def test_paged_attention_float_rows_alone(hq, hkv, d, page, window, split_keys):
    """The float engine: a token's bits do not depend on the tokens that share its workgroup, nor on where a call starts; and a
    value that is not finite reaches exactly the tokens that see it, wherever it lies in a tile of 16 keys."""
    k = kernels(torch.float32)
    n, scale = 150, 1 / math.sqrt(d)
    blocks = (n + page - 1) // page
    q = rnd((n, hq * d), torch.float32, 40)
    k_pages, v_pages = rnd((blocks + 1, hkv, page, d), torch.float32, 41), rnd((blocks + 1, hkv, d, page), torch.float32, 42)
    k_pages[-1], v_pages[-1] = float("nan"), float("nan")
    tail = n - (blocks - 1) * page                       # (behind the last key: never written)
    k_pages[blocks - 1, :, tail:], v_pages[blocks - 1, :, :, tail:] = float("nan"), float("nan")
    table = torch.full((1, blocks + 2), -1, dtype=torch.int32, device="cuda")
    table[0, :blocks] = torch.arange(blocks, dtype=torch.int32)
    splits = -(-n // split_keys) if split_keys else 1
    partial = torch.full((k.attention_partial_numel(n, hq, d, splits),), float("nan"), device="cuda") if split_keys else None

    def run(rows):
        out = torch.full((len(rows), hq * d), float("nan"), device="cuda")
        k.paged_attention(q[rows].contiguous(), k_pages, v_pages, table, torch.zeros(len(rows), dtype=torch.int32, device="cuda"),
                          torch.tensor(rows, dtype=torch.int32, device="cuda"), out, hq, hkv, d, page, scale, window=window,
                          split_keys=split_keys, max_splits=splits, partial=partial)
        return out
    every = list(range(n))
    whole = run(every)
    for rows in ([0], [n - 1], [5], every[3:], every[17:60], every[::-1], every[::7]):
        assert torch.equal(run(rows), whole[rows])
    for bad, at in ((float("inf"), 37), (float("nan"), 64), (float("-inf"), 143)):
        kept = v_pages[at // page, :, :, at % page].clone()
        v_pages[at // page, :, :, at % page] = bad
        hit = torch.tensor([p >= at and (window is None or p - at < window) for p in every])
        got = run(every)
        assert torch.equal(got[~hit], whole[~hit]) and not torch.isfinite(got[hit]).any()
        v_pages[at // page, :, :, at % page] = kept


@pytest.mark.parametrize("hq,hkv,d,page,window,split_keys", [(16, 8, 128, 16, None, 256), (16, 1, 128, 32, 100, 64), (7, 1, 16, 16, None, 0),
                                                             (10, 2, 80, 48, 20, 128), (3, 3, 144, 16, None, 64), (6, 2, 256, 128, 300, 0),
                                                             (5, 1, 192, 64, 1, 64), (8, 2, 64, 16, None, 0)])
def test_paged_attention_float_has_the_general_kernels_bits(hq, hkv, d, page, window, split_keys):
    """Tokens that share a workgroup on the matrix instructions get, to the bit, what the kernel of one token a workgroup gives them
    (reached by queries that do not start on 16 bytes): prompts, single tokens and portions of several requests, in and out of
    order, with pages that end inside a tile."""
    k = kernels(torch.float32)
    lengths, portions = [1, 63, 200, 517, 385], [1, 63, 1, 130, 17]
    blocks = [-(-n // page) for n in lengths]
    order = torch.randperm(sum(blocks), generator=torch.Generator().manual_seed(d)).int()
    k_pages, v_pages = rnd((sum(blocks), hkv, page, d), torch.float32, 50), rnd((sum(blocks), hkv, d, page), torch.float32, 51)
    table = torch.full((len(lengths), max(blocks) + 1), -1, dtype=torch.int32)
    for i, n in enumerate(blocks):
        table[i, :n] = order[sum(blocks[:i]):sum(blocks[:i]) + n]
    rows = [(i, p) for i, (n, m) in enumerate(zip(lengths, portions)) for p in range(n - m, n)]
    splits = -(-max(lengths) // split_keys) if split_keys else 1
    q = rnd((len(rows), hq * d), torch.float32, 52) * 2
    for picked in (list(range(len(rows))), list(range(len(rows)))[::-1], list(range(0, len(rows), 3))):
        partial = torch.full((k.attention_partial_numel(len(picked), hq, d, splits),), float("nan"), device="cuda") if split_keys else None
        got = []
        for spare in (0, 1):
            queries = torch.empty(len(picked) * hq * d + spare, device="cuda")[spare:].view(len(picked), hq * d).copy_(q[picked])
            out = torch.full_like(queries, float("nan"))
            k.paged_attention(queries, k_pages, v_pages, table.cuda(), torch.tensor([rows[i][0] for i in picked], dtype=torch.int32, device="cuda"),
                              torch.tensor([rows[i][1] for i in picked], dtype=torch.int32, device="cuda"), out, hq, hkv, d, page,
                              d ** -0.5, window=window, split_keys=split_keys, max_splits=splits, partial=partial)
            got.append(out)
        assert torch.equal(got[0], got[1])


@pytest.mark.parametrize("dtype", DTYPES)
def test_attention_finds_one_far_key(dtype):
    """One key among a thousand matches the query (scaled so that its score stands out): the
    output must be that key's value, wherever in the pages it lies."""
    k = kernels(dtype)
    hq = hkv = 1
    d, page, L = 64, 16, 1000
    g = torch.Generator().manual_seed(21)
    for far in [0, 15, 16, 63, 64, 511, 512, 998, 999]:
        kk = 0.05 * torch.randn((L, 1, d), generator=g)
        vv = torch.randn((L, 1, d), generator=g)
        q = torch.randn((1, d), generator=g)
        kk[far, 0] = 40 * q[0] / q[0].norm()
        n_blocks = (L + page - 1) // page
        table = torch.arange(n_blocks - 1, -1, -1, dtype=torch.int32)[None, :].contiguous()
        k_pages = torch.zeros((n_blocks, 1, page, d))
        v_pages = torch.zeros((n_blocks, 1, d, page))
        for b in range(n_blocks):
            n = min(page, L - b * page)
            k_pages[table[0, b], 0, :n] = kk[b * page:b * page + n, 0]
            v_pages[table[0, b], 0, :, :n] = vv[b * page:b * page + n, 0].T
        out = torch.empty((1, d), dtype=dtype, device="cuda")
        for split_keys in (0, 128):
            max_splits = (L + split_keys - 1) // split_keys if split_keys else 1
            partial = torch.empty(k.attention_partial_numel(1, 1, d, max_splits), device="cuda") if split_keys else None
            k.paged_attention(q.to(dtype).cuda(), k_pages.to(dtype).cuda(), v_pages.to(dtype).cuda(), table.cuda(),
                              torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([L - 1], dtype=torch.int32).cuda(),
                              out, 1, 1, d, page, 1.0, split_keys=split_keys, max_splits=max_splits, partial=partial)
            torch.testing.assert_close(out.float().cpu()[0], vv[far, 0].to(dtype).float(), atol=3e-2, rtol=3e-2)
            if k.mfma_attention_supported(1, 1, d, page):
                out.fill_(float("nan"))
                one = torch.ones(1, dtype=torch.int32).cuda()
                k.attention_mfma(q.to(dtype).cuda(), k_pages.to(dtype).cuda(), v_pages.to(dtype).cuda(), table.cuda(),
                                 torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([L - 1], dtype=torch.int32).cuda(),
                                 out, torch.zeros(1, dtype=torch.int32).cuda(), one, 1, 1, 1, d, page, 1.0,
                                 split_keys=split_keys, max_splits=max_splits, partial=partial)
                torch.testing.assert_close(out.float().cpu()[0], vv[far, 0].to(dtype).float(), atol=3e-2, rtol=3e-2)


@pytest.mark.parametrize("vocab", [1, 31, 32, 33, 257, 1024, 1025, 151936])
def test_sample_greedy(vocab):
    """Ties -> lowest id; a NaN or infinity -> -1 and the status names the row
    (tests/cuda_ops_tests.cu:408-435)."""
    k = kernels(torch.float32)
    g = torch.Generator().manual_seed(vocab)
    logits = torch.randn((4, vocab), generator=g)
    if vocab > 2:
        logits[1, vocab - 1] = 50.0
        logits[1, vocab // 2] = 50.0
        logits[2, 0] = 60.0
    if vocab > 40:
        logits[3, 37] = float("nan")
    temp = torch.zeros(4).cuda()
    u = torch.zeros(4).cuda()
    tokens = torch.full((4,), -7, dtype=torch.int32).cuda()
    status = torch.zeros(2, dtype=torch.int32).cuda()
    sample(k, logits.cuda(), temp, u, tokens, status)
    got = tokens.cpu().tolist()
    for r in range(4):
        row = logits[r]
        if not torch.isfinite(row).all():
            assert got[r] == -1
        else:
            assert got[r] == int(np.argmax(row.numpy()))
    if vocab > 40:
        assert status.cpu().tolist() == [1, 3]
    else:
        assert status.cpu().tolist() == [0, 2 ** 31 - 1]
    if vocab > 2:
        assert got[1] == vocab // 2 and got[2] == 0


@pytest.mark.parametrize("vocab", [5, 311, 4099, 151936, 1859, 2680, 2769, 146254, 236821])
def test_sample_temperature(vocab):
    """The drawn token's slice of the CDF of softmax(logits / T) (float64) holds u.  Row 1 draws u = 1 - 2^-23:
    in 32-bit its target is the total itself or a rounding below it, and the token must still come from the
    CDF's end (the last five sizes are ones at which the running sums, added in another order, end below it)."""
    from plain.qwen3_plain import temperature_cdf
    k = kernels(torch.float32)
    g = torch.Generator().manual_seed(vocab + 1)
    rows = 64
    logits = 3 * torch.randn((rows, vocab), generator=g)
    temp = torch.rand(rows, generator=g) * 1.5 + 0.2
    u = torch.rand(rows, generator=g)
    u[0], u[1] = 0.0, 0.9999999
    tokens = torch.empty(rows, dtype=torch.int32).cuda()
    status = torch.zeros(2, dtype=torch.int32).cuda()
    sample(k, logits.cuda(), temp.cuda(), u.cuda(), tokens, status)
    got = tokens.cpu().tolist()
    for r in range(rows):
        cdf = temperature_cdf(logits[r].numpy(), float(temp[r]))
        t = got[r]
        lo = cdf[t - 1] if t > 0 else 0.0
        assert lo - 1e-4 <= float(u[r]) <= cdf[t] + 1e-4, (r, t, lo, float(u[r]), cdf[t])


def test_sample_frequencies():
    """Empirical frequencies over many draws follow softmax(logits / T)."""
    k = kernels(torch.float32)
    logits = torch.tensor([0.0, 1.0, 2.0, -1.0, 0.5, 3.0, -2.0])
    temp_value = 0.8
    rows = 20000
    g = torch.Generator().manual_seed(5)
    u = torch.rand(rows, generator=g).cuda()
    tokens = torch.empty(rows, dtype=torch.int32).cuda()
    sample(k, logits[None, :].repeat(rows, 1).cuda().contiguous(), torch.full((rows,), temp_value).cuda(), u, tokens,
           torch.zeros(2, dtype=torch.int32).cuda())
    freq = torch.bincount(tokens.cpu().long(), minlength=7).double() / rows
    want = torch.softmax(logits.double() / temp_value, 0)
    assert (freq - want).abs().max() < 0.015


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("window", [1, 16, 17, 64, 100])
def test_attention_window_edge(dtype, window):
    """The key just outside the window matches the query strongly and must not be seen; then the key
    just inside does and must be seen."""
    k = kernels(dtype)
    d, page, L = 32, 16, 300
    g = torch.Generator().manual_seed(31)
    q = torch.randn((1, d), generator=g)
    for inside in (False, True):
        kk = 0.05 * torch.randn((L, d), generator=g)
        vv = torch.randn((L, d), generator=g)
        hot = L - window + (0 if inside else -1)
        kk[hot] = 40 * q[0] / q[0].norm()
        n_blocks = (L + page - 1) // page
        table = torch.arange(n_blocks, dtype=torch.int32)[None, :].contiguous()
        k_pages = torch.zeros((n_blocks, 1, page, d))
        k_pages.view(-1, d)[:L] = kk
        rows = torch.zeros((n_blocks * page, d))
        rows[:L] = vv
        v_pages = rows.view(n_blocks, 1, page, d).transpose(2, 3).contiguous()
        out = torch.empty((1, d), dtype=dtype, device="cuda")
        k.paged_attention(q.to(dtype).cuda(), k_pages.to(dtype).cuda(), v_pages.to(dtype).cuda(), table.cuda(),
                          torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([L - 1], dtype=torch.int32).cuda(),
                          out, 1, 1, d, page, 1.0, window=window)
        lo = L - window
        want = plain_attention(q.to(dtype).double(), kk[:, None, :].to(dtype).double(), vv[:, None, :].to(dtype).double(),
                               1.0, window)
        torch.testing.assert_close(out.double().cpu(), want, **tol(dtype))
        close_to_hot = (out.float().cpu()[0] - vv[hot].to(dtype).float()).abs().max() < 0.05
        assert bool(close_to_hot) == inside, (window, inside, lo)
        if k.mfma_attention_supported(1, 1, d, page):
            out.fill_(float("nan"))
            k.attention_mfma(q.to(dtype).cuda(), k_pages.to(dtype).cuda(), v_pages.to(dtype).cuda(), table.cuda(),
                             torch.zeros(1, dtype=torch.int32).cuda(), torch.tensor([L - 1], dtype=torch.int32).cuda(),
                             out, torch.zeros(1, dtype=torch.int32).cuda(), torch.ones(1, dtype=torch.int32).cuda(),
                             1, 1, 1, d, page, 1.0, window=window)
            torch.testing.assert_close(out.double().cpu(), want, **tol(dtype))
            assert bool((out.float().cpu()[0] - vv[hot].to(dtype).float()).abs().max() < 0.05) == inside


@pytest.mark.parametrize("mnk", [(1, 48, 64), (8, 3072, 1024), (17, 100, 76), (40, 208, 80), (64, 136, 264),
                                 (3, 56, 192), (16, 40, 4160), (13, 72, 2048)])
def test_gemm_gated_silu(mnk):
    """The feed-forward's activation fused into its first projection (few rows, bfloat16):
    silu(a Wgate^T) * (a Wup^T) with the sums kept in 32-bit until the product."""
    from mini_llm_runtime_amd.kernels import Kernels
    m, n, kk = mnk
    k = Kernels(torch.bfloat16, library_gemm=False)
    assert k.gated_silu_fused(m) and not k.gated_silu_fused(65)
    assert kernels(torch.bfloat16).gated_silu_fused(16) and not kernels(torch.bfloat16).gated_silu_fused(17)
    # with the library at hand, more rows stay here only while the inner size is small
    assert kernels(torch.bfloat16).gated_silu_fused(64, 1024) and not kernels(torch.bfloat16).gated_silu_fused(33, 2048)
    a = rnd((m, kk), torch.bfloat16, 50)
    w = rnd((2 * n, kk), torch.bfloat16, 51, 0.3)
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_gated_silu(a, w, out)
    g = a.double() @ w.double()[:n].T
    u = a.double() @ w.double()[n:].T
    want = g / (1 + torch.exp(-g)) * u
    torch.testing.assert_close(out.double(), want, atol=2e-2 * float(want.abs().max()), rtol=2e-2)


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shape", [(4, 2, 128, 16), (6, 3, 48, 32), (16, 8, 64, 16), (3, 1, 16, 16), (2, 2, 256, 64)])
@pytest.mark.parametrize("layout", [([90, 10], [37, 0]), ([96, 16], [32, 8]), ([64, 3, 40], [0, 5, 16])])
def test_qk_norm_rope_kv_many_rows(dtype, shape, layout):
    """Whole prompt portions (the many-row variants of the kernels): consecutive positions of a few requests,
    starting inside a page, at a page's edge and at multiples of eight."""
    hq, hkv, d, page = shape
    k = kernels(dtype)
    counts, starts = layout
    m = sum(counts)
    n_req = len(counts)
    positions = torch.tensor([starts[s] + i for s in range(n_req) for i in range(counts[s])], dtype=torch.int32)
    slots = torch.tensor([s for s in range(n_req) for _ in range(counts[s])], dtype=torch.int32)
    max_blocks = 16
    n_pages = n_req * max_blocks
    perm = torch.randperm(n_pages, generator=torch.Generator().manual_seed(3)).to(torch.int32)
    table = perm.view(n_req, max_blocks).contiguous()
    qkv = rnd((m, (hq + 2 * hkv) * d), dtype, 60)
    qw, kw = rnd((d,), torch.float32, 61) + 1, rnd((d,), torch.float32, 62) + 1
    eps, base = 1e-6, 10000.0
    rope = rope_table(256, d, base)
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype, device="cuda")
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype, device="cuda")
    q_out = torch.empty((m, hq * d), dtype=dtype, device="cuda")
    k.qk_norm_rope_kv(qkv, q_out, k_pages, v_pages, table.cuda(), slots.cuda(), positions.cuda(), qw, kw, eps, rope,
                      hq, hkv, d, page)
    x = qkv.double().cpu()
    q = x[:, :hq * d].view(m, hq, d)
    kk = x[:, hq * d:(hq + hkv) * d].view(m, hkv, d)

    def norm(t, w):
        return t * torch.rsqrt((t * t).mean(-1, keepdim=True) + eps) * w.double().cpu()
    q_want = plain_rope(norm(q, qw), positions, base)
    k_want = plain_rope(norm(kk, kw), positions, base)
    torch.testing.assert_close(q_out.double().cpu().view(m, hq, d), q_want, **tol(dtype))
    kp, vp = k_pages.cpu(), v_pages.cpu()
    for i in range(m):
        p, s = int(positions[i]), int(slots[i])
        pg = int(table[s, p // page])
        torch.testing.assert_close(kp[pg, :, p % page].double(), k_want[i], **tol(dtype))
        assert torch.equal(vp[pg, :, :, p % page], qkv[i, (hq + hkv) * d:].view(hkv, d).cpu())
    written = sum(counts) * hkv * d
    assert int((~torch.isnan(kp.float())).sum()) == written and int((~torch.isnan(vp.float())).sum()) == written


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("width", [8, 72, 1024, 2048, 2056, 76])
def test_add_rmsnorm_many_rows(dtype, width):
    k = kernels(dtype)
    rows = 130
    h0 = rnd((rows, width), torch.float32, 70, 2.0)
    delta = rnd((rows, width), dtype, 71)
    w = rnd((width,), torch.float32, 72)
    x = h0.double() + delta.double()
    want = x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double()
    h = h0.clone()
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, delta, w, out, 1e-6)
    torch.testing.assert_close(h.double(), x, atol=1e-6, rtol=1e-6)
    torch.testing.assert_close(out.double(), want, **tol(dtype))
    idx = torch.arange(rows - 1, -1, -1, dtype=torch.int32).cuda()[:100].contiguous()
    h = h0.clone()
    out = torch.empty((100, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, delta, w, out, 1e-6, rows=idx, write_h=False)
    assert torch.equal(h, h0)
    torch.testing.assert_close(out.double(), want[idx.long()], **tol(dtype))
    out = torch.empty((rows, width), dtype=dtype, device="cuda")
    k.add_rmsnorm(h, None, w, out, 1e-6)
    x = h0.double()
    torch.testing.assert_close(out.double(), x * torch.rsqrt((x * x).mean(-1, keepdim=True) + 1e-6) * w.double(), **tol(dtype))


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("inter", [8, 104, 3072])
def test_silu_mul_wide(dtype, inter):
    k = kernels(dtype)
    gate_up = rnd((70, 2 * inter), dtype, 80, 3.0)
    act = torch.empty((70, inter), dtype=dtype, device="cuda")
    k.silu_mul(gate_up, act)
    g, u = gate_up.double()[:, :inter], gate_up.double()[:, inter:]
    torch.testing.assert_close(act.double(), g / (1 + torch.exp(-g)) * u, **tol(dtype))


@pytest.mark.parametrize("rows,width", [(1, 64), (8, 1024), (16, 100), (5, 97), (3, 4096)])
def test_rows_prenorm(rows, width):
    """The first half of a norm that is handed to the projection after it: h += delta, out = bf16(h * w) without
    the scale, and the rows' sums of squares."""
    k = kernels(torch.bfloat16)
    h0 = rnd((rows, width), torch.float32, 94, 2.0)
    delta = rnd((rows, width), torch.bfloat16, 95)
    nw = rnd((width,), torch.float32, 96) + 1
    for d in (delta, None):
        h = h0.clone()
        out = torch.full((rows, width), float("nan"), dtype=torch.bfloat16, device="cuda")
        ss = torch.full((rows, 1), float("nan"), device="cuda")
        k.rows_prenorm(h, d, nw, out, ss)
        x = h0.double() + (d.double() if d is not None else 0)
        torch.testing.assert_close(h.double(), x, atol=1e-6, rtol=1e-6)
        torch.testing.assert_close(out.double(), (x * nw.double()).to(torch.bfloat16).double(), atol=0, rtol=2 ** -7)
        torch.testing.assert_close(ss[:, 0].double(), (x * x).sum(-1), rtol=1e-5, atol=1e-5)


@pytest.mark.parametrize("gated", [False, True])
@pytest.mark.parametrize("mnk,parts", [((1, 48, 64), 1), ((8, 4096, 1024), 64), ((16, 100, 1024), 3), ((5, 208, 96), 6),
                                       ((3, 40, 4096), 256), ((7, 24, 32), 2), ((2, 50, 100), 7), ((16, 333, 2048), 128),
                                       ((4, 48, 8320), 520), ((6, 32, 2096), 131), ((9, 64, 5120), 320)])
def test_projection_after_a_handed_over_norm(mnk, parts, gated):
    """`gemm_prenormed`: the rows' scale rsqrt(sum of the partial sums / K + eps), applied to the finished sums
    of x . w^T (or inside the gated activation), equals the projection of the normed rows.  The partial sums are
    read four a load where their number is a multiple of four and they start at a multiple of 16 bytes, else
    one a load, in rounds of four loads (520 and 131 parts: more than one round)."""
    m, n, kk = mnk
    k = kernels(torch.bfloat16)
    assert k.handoff_supported(m) and not k.handoff_supported(17) and not kernels(torch.float32).handoff_supported(m)
    xf = rnd((m, kk), torch.float32, 90, 2.0)
    nw = rnd((kk,), torch.float32, 92) + 1
    x = (xf * nw).to(torch.bfloat16)
    # the rows' sums of squares, cut into parts of any sizes (some of them zero)
    cuts = torch.linspace(0, kk, parts + 1).long().tolist()
    ss = torch.stack([(xf[:, a:b].double() ** 2).sum(-1) for a, b in zip(cuts, cuts[1:])], dim=1).float().contiguous()
    w = rnd(((2 if gated else 1) * n, kk), torch.bfloat16, 93, 0.2)
    eps = 1e-5
    out = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_prenormed(x, ss, eps, w, out, gated=gated)
    scale = torch.rsqrt((xf.double() ** 2).mean(-1, keepdim=True) + eps)
    if gated:
        g, u = scale * (x.double() @ w.double()[:n].T), scale * (x.double() @ w.double()[n:].T)
        want = g / (1 + torch.exp(-g)) * u
    else:
        want = scale * (x.double() @ w.double().T)
    torch.testing.assert_close(out.double(), want, atol=1e-2 * float(want.abs().max()), rtol=1e-2)
    # a row's result does not depend on the rows beside it
    if m > 1:
        one = torch.full((1, n), float("nan"), dtype=torch.bfloat16, device="cuda")
        k.gemm_prenormed(x[m - 1:].contiguous(), ss[m - 1:].contiguous(), eps, w, one, gated=gated)
        assert torch.equal(one[0], out[m - 1])
    # the same sums at an address that is no multiple of 16 bytes (read one a load)
    shifted = torch.empty(m * parts + 1, dtype=torch.float32, device="cuda")[1:].view(m, parts)
    shifted.copy_(ss)
    assert shifted.data_ptr() % 16 == 4
    again = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_prenormed(x, shifted, eps, w, again, gated=gated)
    torch.testing.assert_close(again.double(), want, atol=1e-2 * float(want.abs().max()), rtol=1e-2)


@pytest.mark.parametrize("mnk", [(1, 64, 48), (8, 1024, 2048), (16, 1024, 3072), (5, 96, 208), (3, 4096, 4096), (7, 50, 96),
                                 (2, 97, 100), (16, 40, 64), (9, 4096, 12288), (8, 5120, 2048), (3, 4100, 2048),
                                 (16, 5120, 8192)])
def test_projection_that_adds_into_the_residual_stream(mnk):
    """`gemm_residual`: h += a . w^T in 32-bit; with a norm to follow also bf16(h * next_w) and partial sums of
    squares of the new h: per row and strip of 16 columns or, where a workgroup owns two strips side by side
    (the last three shapes), per row and workgroup, the parts beyond the workgroups zero."""
    m, n, kk = mnk
    k = kernels(torch.bfloat16)
    a = rnd((m, kk), torch.bfloat16, 97)
    w = rnd((n, kk), torch.bfloat16, 98, 0.2)
    h0 = rnd((m, n), torch.float32, 99, 2.0)
    nw = rnd((n,), torch.float32, 100) + 1
    want_h = h0.double() + a.double() @ w.double().T
    tol_h = dict(atol=2e-5 * float(want_h.abs().max()) * max(1, kk // 512), rtol=1e-5)
    h = h0.clone()
    k.gemm_residual(a, w, h)
    torch.testing.assert_close(h.double(), want_h, **tol_h)
    h2 = h0.clone()
    parts = k.handoff_parts(n)
    x = torch.full((m, n), float("nan"), dtype=torch.bfloat16, device="cuda")
    ss = torch.full((m, parts), float("nan"), device="cuda")
    k.gemm_residual(a, w, h2, nw, x, ss)
    assert torch.equal(h2, h)
    torch.testing.assert_close(x.double(), (h.double() * nw.double()).to(torch.bfloat16).double(), atol=0, rtol=2 ** -7)
    padded = torch.zeros((m, parts * 16), dtype=torch.float64, device="cuda")
    padded[:, :n] = h.double() ** 2
    if n in (5120, 4100):
        used = int((ss != 0).any(dim=0).sum())              # a part a workgroup: fewer than strips of 16, a prefix
        assert bool(torch.isfinite(ss).all()) and parts // 2 <= used < parts and bool((ss[:, used:] == 0).all())
        torch.testing.assert_close(ss.double().sum(-1), padded.sum(-1), rtol=1e-5, atol=1e-6)
    else:
        torch.testing.assert_close(ss.double(), padded.view(m, parts, 16).sum(-1), rtol=1e-5, atol=1e-6)
    # the two halves together are the norm: the next projection on (x, ss) gives rmsnorm(h) . w2^T
    w2 = rnd((64, n), torch.bfloat16, 101, 0.2)
    out = torch.full((m, 64), float("nan"), dtype=torch.bfloat16, device="cuda")
    k.gemm_prenormed(x, ss, 1e-6, w2, out)
    hn = h.double() * torch.rsqrt((h.double() ** 2).mean(-1, keepdim=True) + 1e-6) * nw.double()
    want = hn @ w2.double().T
    torch.testing.assert_close(out.double(), want, atol=2e-2 * float(want.abs().max()), rtol=2e-2)


def test_prompt_portion_beyond_the_page_cache_of_a_workgroup():
    """A portion of 70 tokens at the end of a context of 33 000 keys: more pages than a workgroup of the
    32x32-tile kernel keeps, so the keys must be split; unsplit the call is refused."""
    from mini_llm_runtime_amd.kernels.ops import KernelError
    dtype = torch.bfloat16
    k = kernels(dtype)
    hq, hkv, d, page, L, n = 2, 1, 64, 16, 33000, 70
    g = torch.Generator().manual_seed(77)
    kk = torch.randn((L, hkv, d), generator=g).to(dtype)
    vv = torch.randn((L, hkv, d), generator=g).to(dtype)
    blocks = (L + page - 1) // page
    perm = torch.randperm(blocks, generator=g)
    table = perm.to(torch.int32)[None, :].contiguous()
    k_pages = torch.zeros((blocks, hkv, page, d), dtype=dtype)
    v_pages = torch.zeros((blocks, hkv, d, page), dtype=dtype)
    pad = blocks * page - L
    kp = torch.cat([kk, torch.zeros((pad, hkv, d), dtype=dtype)]).view(blocks, page, hkv, d)
    vp = torch.cat([vv, torch.zeros((pad, hkv, d), dtype=dtype)]).view(blocks, page, hkv, d)
    k_pages[perm] = kp.permute(0, 2, 1, 3)
    v_pages[perm] = vp.permute(0, 2, 3, 1)
    q = (torch.randn((n, hq, d), generator=g) * 2).to(dtype)
    pos = torch.arange(L - n, L, dtype=torch.int32).cuda()
    slots = torch.zeros(n, dtype=torch.int32).cuda()
    first = torch.tensor([0, 64], dtype=torch.int32).cuda()
    count = torch.tensor([64, 6], dtype=torch.int32).cuda()
    out = torch.full((n, hq * d), float("nan"), dtype=dtype, device="cuda")
    args = (q.view(n, hq * d).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), slots, pos, out, first, count, 2,
            hq, hkv, d, page, 1 / math.sqrt(d))
    with pytest.raises(KernelError):
        k.attention_tiles(*args, max_context=L)
    split = 16384
    splits = (L + split - 1) // split
    part = torch.full((k.attention_partial_numel(n, hq, d, splits),), float("nan"), device="cuda")
    k.attention_tiles(*args, max_context=L, split_keys=split, max_splits=splits, partial=part)
    got = out.double().cpu().view(n, hq, d)
    for i in (0, 1, 31, 63, 64, 69):
        want = plain_attention(q[i].double(), kk[:L - n + i + 1].double(), vv[:L - n + i + 1].double(), 1 / math.sqrt(d), None)
        torch.testing.assert_close(got[i], want, **tol(dtype))


@pytest.mark.parametrize("case", [
    # (q heads, kv heads, head_dim, page, context lengths of the requests, window, split_keys, norm, rotation)
    (16, 8, 128, 16, [1, 2, 17, 300, 4096], None, 512, True, True),
    (4, 4, 64, 16, [1, 33, 64, 65, 130], None, 0, True, True),
    (8, 2, 64, 32, [5, 100, 257], 40, 64, True, True),
    (6, 1, 192, 16, [1, 70], None, 0, False, True),
    (2, 1, 256, 16, [129, 1], 1, 64, True, False),
    (32, 8, 128, 64, [513, 512, 511], 512, 256, True, True),
    # (heads above 128 channels, where a lane holds two rotation pairs: cases in which the two ways once differed
    # in a key's last bit, the compiler having fused the products and sums of the two kernels differently)
    (10, 5, 256, 32, [2078, 867, 853, 202], 441, 0, True, True),
    (15, 3, 192, 128, [1, 246, 75, 83, 345, 236, 609], None, 64, True, True),
    (64, 8, 256, 16, [2270, 123, 1915, 575, 687], None, 0, False, True),
])
def test_decode_attention_that_norms_rotates_and_caches_itself(case):
    """Every request brings one new token.  The fused pair of launches against the separate ones (per-head
    norm + rotation + cache write, then attention): the same output within bfloat16 rounding, the same key and
    value in the cache bit for bit, nothing else in the cache touched; and against the plain attention."""
    hq, hkv, d, page, lengths, window, split_keys, with_norm, with_rope = case
    dtype = torch.bfloat16
    k = kernels(dtype)
    gen = torch.Generator().manual_seed(41)
    n = len(lengths)
    max_len = max(lengths)
    max_blocks = (max_len + page - 1) // page
    n_pages = sum((L + page - 1) // page for L in lengths) + 3
    perm = torch.randperm(n_pages, generator=gen).tolist()
    table = torch.full((n, max_blocks), -1, dtype=torch.int32)
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype)
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype)
    keys, values = [], []
    for s, L in enumerate(lengths):
        kk = torch.randn((L - 1, hkv, d), generator=gen).to(dtype)
        vv = torch.randn((L - 1, hkv, d), generator=gen).to(dtype)
        keys.append(kk)
        values.append(vv)
        for b in range((L + page - 1) // page):
            pg = perm.pop()
            table[s, b] = pg
            cnt = max(0, min(page, L - 1 - b * page))
            if cnt:
                k_pages[pg, :, :cnt] = kk[b * page:b * page + cnt].transpose(0, 1)
                v_pages[pg, :, :, :cnt] = vv[b * page:b * page + cnt].permute(1, 2, 0)
    qkv = (torch.randn((n, (hq + 2 * hkv) * d), generator=gen) * 1.5).to(dtype).cuda()
    qw = (1 + 0.2 * torch.randn(d, generator=gen)).cuda() if with_norm else None
    kw = (1 + 0.2 * torch.randn(d, generator=gen)).cuda() if with_norm else None
    eps, base, scale = 1e-5, 10000.0, 1 / math.sqrt(d)
    rope = rope_table(max_len, d, base).cuda() if with_rope else None
    slots = torch.arange(n, dtype=torch.int32).cuda()
    pos = torch.tensor([L - 1 for L in lengths], dtype=torch.int32).cuda()
    first = torch.arange(n, dtype=torch.int32).cuda()
    ones = torch.ones(n, dtype=torch.int32).cuda()
    max_splits = (max_len + split_keys - 1) // split_keys if split_keys else 1
    partial = torch.full((k.attention_partial_numel(n, hq, d, max_splits),), float("nan"), device="cuda")
    # the separate launches
    k1, v1 = k_pages.clone().cuda(), v_pages.clone().cuda()
    q1 = torch.empty((n, hq * d), dtype=dtype, device="cuda")
    k.qk_norm_rope_kv(qkv, q1, k1, v1, table.cuda(), slots, pos, qw, kw, eps, rope, hq, hkv, d, page)
    out1 = torch.full((n, hq * d), float("nan"), dtype=dtype, device="cuda")
    k.attention_mfma(q1, k1, v1, table.cuda(), slots, pos, out1, first, ones, n, hq, hkv, d, page, scale, window=window,
                     split_keys=split_keys, max_splits=max_splits, partial=partial if max_splits > 1 else None)
    # the fused ones
    k2, v2 = k_pages.clone().cuda(), v_pages.clone().cuda()
    out2 = torch.full((n, hq * d), float("nan"), dtype=dtype, device="cuda")
    partial.fill_(float("nan"))
    k.attention_decode_fused(qkv, k2, v2, table.cuda(), slots, pos, out2, first, ones, n, hq, hkv, d, page, scale,
                             qw, kw, eps, rope, partial, window=window, split_keys=split_keys, max_splits=max_splits)
    same = lambda x, y: torch.equal(x.view(torch.int16), y.view(torch.int16))     # NaN-filled entries compare too
    assert same(k1, k2) and same(v1, v2)
    torch.testing.assert_close(out2.float(), out1.float(), atol=2e-2, rtol=2e-2)
    # and the plain attention over the cached keys plus the new one, as the separate launches cached it
    for s, L in enumerate(lengths):
        pg, at = table[s, (L - 1) // page].item(), (L - 1) % page
        kk = torch.cat([keys[s], k1[pg, :, at].cpu()[None]]).double()
        vv = torch.cat([values[s], v1[pg, :, :, at].cpu()[None]]).double()
        want = plain_attention(q1[s].double().cpu().view(hq, d), kk, vv, scale, window)
        torch.testing.assert_close(out2[s].double().cpu().view(hq, d), want, **tol(dtype))


@pytest.mark.parametrize("d", [64, 128])
def test_decoding_beyond_the_page_cache_of_a_workgroup(d):
    """One new token behind 66 000 keys in pages of 16 (4125 pages: more than the 4096 ids that a workgroup of
    the single-token kernels keeps), beside a short request: unsplit the calls are refused; with the key ranges
    that the engine forces on such a context both kernels (queries prepared, and the one that norms, rotates and
    caches inside itself) give the plain attention and the same cache.  Random keys would hide a range that is
    skipped among thousands: a key near the start, the last key of the first range, the first of the last range
    and the last cached key are made to stand out, each with a value of its own."""
    from mini_llm_runtime_amd.kernels.ops import KernelError, Kernels
    dtype = torch.bfloat16
    k = kernels(dtype)
    hq, hkv, page = 2, 1, 16
    lengths = [66000, 40]
    assert lengths[0] > Kernels.mfma_longest_context(page)
    gen = torch.Generator().manual_seed(5)
    n, max_len = len(lengths), max(lengths)
    max_blocks = (max_len + page - 1) // page
    n_pages = sum((L + page - 1) // page for L in lengths) + 3
    perm = torch.randperm(n_pages, generator=gen).tolist()
    table = torch.full((n, max_blocks), -1, dtype=torch.int32)
    k_pages = torch.full((n_pages, hkv, page, d), float("nan"), dtype=dtype)
    v_pages = torch.full((n_pages, hkv, d, page), float("nan"), dtype=dtype)
    qkv = (torch.randn((n, (hq + 2 * hkv) * d), generator=gen) * 1.5).to(dtype)
    split_keys = 32768
    marked = [5, split_keys - 1, 2 * split_keys, lengths[0] - 2]
    keys, values = [], []
    for s, L in enumerate(lengths):
        kk = torch.randn((L - 1, hkv, d), generator=gen).to(dtype)
        vv = torch.randn((L - 1, hkv, d), generator=gen).to(dtype)
        if s == 0:
            for j, at in enumerate(marked):            # along the first head's query: a score far above the others'
                kk[at, 0] = (qkv[0, :d].float() * (1.2 + 0.01 * j)).to(dtype)
                vv[at, 0] = 0
                vv[at, 0, j] = 8.0
        keys.append(kk)
        values.append(vv)
        flat_k = torch.cat([kk, torch.full((1, hkv, d), float("nan"), dtype=dtype)])       # (the new token's place)
        flat_v = torch.cat([vv, torch.full((1, hkv, d), float("nan"), dtype=dtype)])
        for b in range((L + page - 1) // page):
            pg = perm.pop()
            table[s, b] = pg
            cnt = min(page, L - b * page)
            k_pages[pg, :, :cnt] = flat_k[b * page:b * page + cnt].transpose(0, 1)
            v_pages[pg, :, :, :cnt] = flat_v[b * page:b * page + cnt].permute(1, 2, 0)
    qkv = qkv.cuda()
    scale = 1 / math.sqrt(d)
    slots = torch.arange(n, dtype=torch.int32).cuda()
    pos = torch.tensor([L - 1 for L in lengths], dtype=torch.int32).cuda()
    first = torch.arange(n, dtype=torch.int32).cuda()
    ones = torch.ones(n, dtype=torch.int32).cuda()
    max_splits = (max_len + split_keys - 1) // split_keys
    partial = torch.full((k.attention_partial_numel(n, hq, d, max_splits),), float("nan"), device="cuda")
    # no norm and no rotation: what is cached is the raw key, so the plain result below needs no second path
    k1, v1 = k_pages.clone().cuda(), v_pages.clone().cuda()
    q1 = torch.empty((n, hq * d), dtype=dtype, device="cuda")
    k.qk_norm_rope_kv(qkv, q1, k1, v1, table.cuda(), slots, pos, None, None, 0.0, None, hq, hkv, d, page)
    out1 = torch.full((n, hq * d), float("nan"), dtype=dtype, device="cuda")
    with pytest.raises(KernelError, match="4096 pages"):
        k.attention_mfma(q1, k1, v1, table.cuda(), slots, pos, out1, first, ones, n, hq, hkv, d, page, scale)
    k.attention_mfma(q1, k1, v1, table.cuda(), slots, pos, out1, first, ones, n, hq, hkv, d, page, scale,
                     split_keys=split_keys, max_splits=max_splits, partial=partial)
    k2, v2 = k_pages.clone().cuda(), v_pages.clone().cuda()
    out2 = torch.full((n, hq * d), float("nan"), dtype=dtype, device="cuda")
    with pytest.raises(KernelError, match="4096 pages"):
        k.attention_decode_fused(qkv, k2, v2, table.cuda(), slots, pos, out2, first, ones, n, hq, hkv, d, page, scale,
                                 None, None, 0.0, None, partial)
    partial.fill_(float("nan"))
    k.attention_decode_fused(qkv, k2, v2, table.cuda(), slots, pos, out2, first, ones, n, hq, hkv, d, page, scale,
                             None, None, 0.0, None, partial, split_keys=split_keys, max_splits=max_splits)
    same = lambda x, y: torch.equal(x.view(torch.int16), y.view(torch.int16))
    assert same(k1, k2) and same(v1, v2)
    own_k = qkv[:, hq * d:(hq + hkv) * d].cpu().view(n, 1, hkv, d)
    own_v = qkv[:, (hq + hkv) * d:].cpu().view(n, 1, hkv, d)
    for s, L in enumerate(lengths):
        kk = torch.cat([keys[s], own_k[s]]).double()
        vv = torch.cat([values[s], own_v[s]]).double()
        want = plain_attention(qkv[s, :hq * d].double().cpu().view(hq, d), kk, vv, scale, None)
        if s == 0:                                   # each marked key carries a visible share of the first head's result
            assert all(float(want[0, j]) > 0.5 for j in range(len(marked))), want[0, :len(marked)]
        for out in (out1, out2):
            torch.testing.assert_close(out[s].double().cpu().view(hq, d), want, **tol(dtype))


def test_bfloat16_widening_and_rounding():
    """Every one of the 65536 bfloat16 patterns widens to the float of the same value (the embedding gather
    is the kernel that does nothing else), and a 32-bit sum that lies exactly between two bfloat16 values
    is rounded to the even one (the projections' epilogue), below and above one, in both signs -- the
    reference checks its 16-bit conversions the same way (tests/core_tests.cpp:244-254,
    tests/cuda_ops_tests.cu:75-101)."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = kernels(torch.bfloat16)
    patterns = torch.arange(65536, dtype=torch.int32).to(torch.int16).view(torch.bfloat16).view(512, 128).cuda()
    ids = torch.arange(512, dtype=torch.int32, device="cuda")
    h = torch.empty((512, 128), dtype=torch.float32, device="cuda")
    k.embed_gather(ids, patterns, h)
    want = patterns.float()
    assert torch.equal(h.view(torch.int32), want.view(torch.int32))          # bit for bit, NaN payloads too
    # sums a0 * 1 + a1 * 1 with a0 a bfloat16 value and a1 half a unit in its last place
    cases = []
    for exponent in (-20, -1, 0, 1, 7, 30):
        for mantissa in (0, 1, 2, 126, 127):
            base = (1.0 + mantissa / 128.0) * 2.0 ** exponent
            half_ulp = 2.0 ** (exponent - 8)
            even = base if mantissa % 2 == 0 else base + 2 * half_ulp
            for sign in (1.0, -1.0):
                cases.append((sign * base, sign * half_ulp, sign * even))
    a = torch.tensor([[c[0], c[1]] for c in cases], dtype=torch.float32)
    assert torch.equal(a.to(torch.bfloat16).float(), a)                      # the summands are exact in bfloat16
    w = torch.ones((8, 2), dtype=torch.bfloat16, device="cuda")
    want = torch.tensor([c[2] for c in cases], dtype=torch.float32)
    for engine in (k, Kernels(torch.bfloat16, library_gemm=False)):
        for rows in (len(cases), 16, 5):                                     # many rows (the library, or tiles) and few
            out = torch.empty((rows, 8), dtype=torch.bfloat16, device="cuda")
            engine.gemm(a[:rows].to(torch.bfloat16).cuda(), w, out)
            assert torch.equal(out.float().cpu(), want[:rows, None].expand(rows, 8)), rows


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [3, 96])
def test_a_position_beyond_the_block_table_has_no_page(dtype, rows):
    """The engine never asks for it (the cache manager bounds a request's length by its row of the table); a
    caller of the kernels that does gets what a missing page gives: the query is normed and rotated, nothing
    is cached, and no kernel reads past the table's row.  Few rows (the general kernel) and many (the vector
    kernel and its transposing value writer)."""
    hq, hkv, d, page, max_blocks = 4, 2, 64, 16, 2
    k = kernels(dtype)
    inside = max_blocks * page                                         # 32 positions have a page
    positions = torch.tensor([30 + 3 * (i // 2) for i in range(rows)], dtype=torch.int32)      # 30, 30, 33, 33, ...
    slots = torch.tensor([i % 2 for i in range(rows)], dtype=torch.int32)
    seen = {(int(slots[i]), int(positions[i])): i for i in range(rows)}         # (every position of a slot once)
    assert len(seen) == rows
    table = torch.tensor([[3, 0], [1, 2]], dtype=torch.int32)
    qkv = rnd((rows, (hq + 2 * hkv) * d), dtype, 70)
    qw, kw = rnd((d,), torch.float32, 71) + 1, rnd((d,), torch.float32, 72) + 1
    rope = rope_table(256, d, 10000.0)
    k_pages = torch.full((4, hkv, page, d), float("nan"), dtype=dtype, device="cuda")
    v_pages = torch.full((4, hkv, d, page), float("nan"), dtype=dtype, device="cuda")
    q_out = torch.full((rows, hq * d), float("nan"), dtype=dtype, device="cuda")
    k.qk_norm_rope_kv(qkv, q_out, k_pages, v_pages, table.cuda(), slots.cuda(), positions.cuda(), qw, kw, 1e-6, rope,
                      hq, hkv, d, page)
    assert bool(torch.isfinite(q_out.float()).all())
    cached = sum(1 for (s, p) in seen if p < inside)
    kp, vp = k_pages.cpu().float(), v_pages.cpu().float()
    assert int((~torch.isnan(kp)).sum()) == cached * hkv * d and int((~torch.isnan(vp)).sum()) == cached * hkv * d
    for (s, p), i in seen.items():
        if p < inside:
            assert torch.equal(v_pages[int(table[s, p // page]), :, :, p % page].cpu(),
                               qkv[i, (hq + hkv) * d:].view(hkv, d).cpu())


def test_models_with_a_router_do_not_turn_on_timed_plans():
    """A large product of a row count whose library plan is chosen by timing: the library's for a model without a router, and by the rule
    of any other row count, so in one order of sums, for a model with one."""
    from mini_llm_runtime_amd.kernels import Kernels
    plain, routed = Kernels(torch.bfloat16), Kernels(torch.bfloat16, routed=True)
    for n, kk in [(2048, 8448), (4000, 4096), (8000, 2048)]:
        assert not plain.wide_product(2048, n, kk)
        assert routed.wide_product(2048, n, kk) == routed.wide_product(2047, n, kk)
    assert plain.wide_product(2048, 2048, 2048) and routed.wide_product(2048, 2048, 2048)


@pytest.mark.parametrize("m,n,kk,act,taken", [
    # (time of the many-row kernel over the library's and the activation's launch, where both were measured)
    (900, 25600, 5120, "silu", False), (777, 12288, 4096, "silu", False),        # 1.19 and 1.27 while the epilogue's time was a gain
    (2048, 12288, 4096, "silu", False), (2048, 4096, 12288, None, False), (512, 5120, 8192, None, False),    # 1.08, 1.15 and 1.22: plans that were timed
    (128, 792, 11776, None, False), (97, 48000, 3008, None, False),              # 1.85 and 1.11: few outputs of a long k, a long weight
    (64, 31368, 2176, None, False), (40, 29528, 3328, None, False), (24, 36000, 576, None, False),           # 1.06, 1.04: long weights beside few rows
    (2048, 1024, 3072, None, True), (2048, 3072, 1024, "silu", True), (1533, 5120, 25600, None, True),       # 0.92, 0.90 and 0.69
    (32, 12288, 1024, "silu", True), (64, 6144, 2048, None, True), (32, 4096, 8192, None, True)])
def test_the_rule_between_the_kernel_and_the_library_follows_its_measurements(m, n, kk, act, taken):
    assert kernels(torch.bfloat16).wide_product(m, n, kk, act) == taken
