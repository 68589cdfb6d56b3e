"""The attention of prompt portions with a mask rule on the 32 x 32 matrix tiles, and latent attention whose portions make
keys and values of their own, against the same formulas in 64 bits."""
import pytest
import torch

pytestmark = pytest.mark.gpu
BF16 = torch.bfloat16


def attended(q, keys, values, positions, mask, size, keep, sink, scale, cap):
    """q [M, H, D] at `positions` over keys [T, G, D], values [T, G, V]: float64 [M, H, V]."""
    q, keys, values = q.double(), keys.double(), values.double()
    H, G, T = q.shape[1], keys.shape[1], keys.shape[0]
    p, j = positions[:, None].cpu(), torch.arange(T)[None]
    seen = j <= p
    if mask == "window":
        seen &= (p - j < size) | (j < keep)
    elif mask == "chunk":
        seen &= (j // size == p // size) | (j < keep)
    out = []
    for h in range(H):
        s = (q[:, h] @ keys[:, h // (H // G)].T) * scale
        s = s if cap is None else cap * torch.tanh(s / cap)
        s = s.masked_fill(~seen, -torch.inf)
        if sink is not None:
            s = torch.cat([s, sink[h].double().expand(s.shape[0], 1)], 1)
        out.append(torch.softmax(s, 1)[:, :T] @ values[:, h // (H // G)])
    return torch.stack(out, 1)


def rounded(g, *shape, scale=1.0):
    return (torch.randn(shape, generator=g) * scale).to(BF16)


def ints(values):
    return torch.tensor(values, dtype=torch.int32, device="cuda")


@pytest.mark.parametrize("mask,size,keep", [(None, 0, 0), ("window", 37, 0), ("window", 90, 70), ("window", 64, 5), ("window", 1, 0),
                                            ("chunk", 24, 0), ("chunk", 64, 0)])
@pytest.mark.parametrize("heads,kv,dim,vdim,page,cap,with_sink", [(8, 2, 128, 128, 16, None, True), (3, 3, 64, 64, 32, 20.0, False),
                                                                  (20, 1, 64, 128, 128, None, False), (5, 1, 128, 128, 64, 6.0, True)])
def test_portions_with_a_mask(mask, size, keep, heads, kv, dim, vdim, page, cap, with_sink):
    """A portion that starts a prompt and one from the middle of another in one launch, whose lengths fill no group, block or
    page; unwritten places and pages that a window has given back hold NaN."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(BF16)
    g = torch.Generator().manual_seed(heads * 100 + size)
    lengths, begins = [91, 333], [0, 201]
    keys, values = [rounded(g, n, kv, dim, scale=0.5) for n in lengths], [rounded(g, n, kv, vdim) for n in lengths]
    blocks = [-(-n // page) for n in lengths]
    order = torch.randperm(sum(blocks) + 1, generator=g).tolist()
    k_pages = torch.full((sum(blocks) + 1, kv, page, dim), float("nan"), dtype=BF16)
    v_pages = torch.full((sum(blocks) + 1, kv, page, vdim), float("nan"), dtype=BF16)
    table = torch.full((2, max(blocks) + 1), -1, dtype=torch.int32)
    for r in range(2):
        first_seen = begins[r] - size + 1 if mask == "window" else begins[r] // size * size if mask else 0
        for b in range(blocks[r]):
            if (b + 1) * page <= first_seen and b * page >= keep:
                continue                                       # (given back)
            page_id = order.pop()
            table[r, b] = page_id
            part = slice(b * page, min((b + 1) * page, lengths[r]))
            k_pages[page_id, :, :part.stop - part.start] = keys[r][part].transpose(0, 1)
            v_pages[page_id, :, :part.stop - part.start] = values[r][part].transpose(0, 1)
    positions = torch.cat([torch.arange(b, n) for b, n in zip(begins, lengths)])
    rows = [n - b for b, n in zip(begins, lengths)]
    slots = [0] * rows[0] + [1] * rows[1]
    q = rounded(g, sum(rows), heads, dim, scale=0.5)
    sink = torch.randn(heads, generator=g) if with_sink else None
    want = torch.cat([attended(q[:rows[0]], keys[0], values[0], positions[:rows[0]], mask, size, keep, sink, 0.25, cap),
                      attended(q[rows[0]:], keys[1], values[1], positions[rows[0]:], mask, size, keep, sink, 0.25, cap)])
    per = heads // kv
    head_block = 1
    while head_block < per:
        head_block *= 2
    for columns in (64, 128):
        tokens = columns // head_block
        first = [at for r, base in ((0, 0), (1, rows[0])) for at in range(base, base + rows[r], tokens)]
        count = [min(tokens, (rows[0] if at < rows[0] else sum(rows)) - at) for at in first]
        out = torch.full((sum(rows), heads * vdim), float("nan"), dtype=BF16, device="cuda")
        assert k.portion_attention_supported(heads, kv, dim, vdim, dim, vdim, page, mask, size, 400, keep)
        k.portion_attention(q.reshape(sum(rows), -1).cuda(), k_pages.cuda(), v_pages.cuda(), table.cuda(), ints(slots), positions.int().cuda(),
                            None if sink is None else sink.cuda(), out, ints(first), ints(count), len(first), columns, head_block, heads,
                            kv, dim, vdim, page, 0.25, mask, size, 400, keep, cap)
        # probabilities and the result are rounded to 2^-9 each, of values of size 1
        torch.testing.assert_close(out.double().cpu().view(want.shape), want, atol=1.5e-2, rtol=1e-2)


@pytest.mark.parametrize("mask,size", [(None, 0), ("window", 100), ("window", 7), ("chunk", 64)])
@pytest.mark.parametrize("heads,begin,rows", [(3, 0, 250), (1, 130, 120), (2, 257, 65)])
def test_portions_with_keys_in_two_parts(mask, size, heads, begin, rows):
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(BF16)
    g = torch.Generator().manual_seed(heads + begin + size)
    total = begin + rows
    plain, turned, values = rounded(g, total, heads, 128, scale=0.4), rounded(g, total, 64, scale=0.4), rounded(g, total, heads, 128)
    q = rounded(g, rows + 3, heads, 192, scale=0.4)            # (the portion stands behind three other rows)
    sink = torch.randn(heads, generator=g)
    positions = torch.cat([torch.zeros(3, dtype=torch.long), torch.arange(begin, total)])
    want = attended(q[3:], torch.cat([plain, turned[:, None].expand(total, heads, 64)], 2), values, positions[3:], mask, size, 0, sink, 0.2, None)
    first = 0 if mask is None else max(0, begin - size + 1) if mask == "window" else begin // size * size
    first = first // 64 * 64
    on_gpu = q.cuda()
    for columns in (64, 128):
        out = torch.full((rows + 3, heads * 128), float("nan"), dtype=BF16, device="cuda")
        k.portion_attention_split(on_gpu[:, :, :128], on_gpu[:, :, 128:], plain[first:].reshape(-1, heads * 128).cuda(), turned[first:].cuda(),
                                  values[first:].reshape(-1, heads * 128).cuda(), torch.zeros(rows + 3, dtype=torch.int32, device="cuda"),
                                  positions.int().cuda(), sink.cuda(), out, 3, rows, first, columns, heads, 0.2, mask, size)
        assert torch.isnan(out[:3].float()).all()
        torch.testing.assert_close(out[3:].double().cpu().view(want.shape), want, atol=1.5e-2, rtol=1e-2)


@pytest.mark.parametrize("window", [70, 1000])
def test_latent_portions_of_a_model(tmp_path, window, monkeypatch):
    """A model whose latent attention has the sizes of that path, in every way of cutting: portions that make their keys (64
    tokens and more, from the start and from the middle, beside single tokens and short portions), against the plain
    implementation."""
    from helpers import compare, make_requests, plain_logits, portions, run_steps, whole
    from plain import pamunex_plain as P
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Runner
    from mini_llm_runtime_amd.kernels import Kernels
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    latent = dict(type="latent_attention", mlp=None, mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=48, scale=192 ** -0.5,
                                                                rot=dict(dims=64, base=10000.0), mask=dict(size=window)))
    cfg = dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=[latent, latent])
    folder = str(tmp_path / "model")
    write_random_model(folder, config_from_dict(cfg), seed=3, matrix_std=0.12, norm_std=0.2)
    requests = make_requests(97, [150, 64, 201, 9], seed=2)
    want = plain_logits(P.PlainPamunex(folder), requests)
    part = lambda rid, lo, hi: dict(id=rid, tokens=requests[rid][lo:hi], want=list(range(hi - lo)))
    beside = [dict(step=0, entries=[part("r0", 0, 70), part("r3", 0, 5)], end=[]),
              dict(step=1, entries=[part("r3", 5, 6), part("r0", 70, 71), part("r2", 0, 130), part("r1", 0, 64)], end=["r1"]),
              dict(step=2, entries=[part("r3", 6, 9), part("r2", 130, 201), part("r0", 71, 150)], end=["r0", "r2", "r3"])]
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 0)
    calls = []
    original = Kernels.portion_attention_split
    monkeypatch.setattr(Kernels, "portion_attention_split", lambda self, *a, **kw: calls.append(a) or original(self, *a, **kw))
    model = DecoderModel.load(folder, BF16)
    for cut in (whole(requests), portions(requests, (100, 65, 64, 7)), beside):
        calls.clear()
        runner = Runner(model, max_tokens=640, max_slots=4, max_length=256, max_batch_tokens=512, page_size=16)
        compare(run_steps(runner, cut), want, "bfloat16")
        assert calls, "no portion made its keys"
        assert runner.workspace.unplanned_bytes() == 0
    # a budget without room for the scratch memory of long portions: the runner is built all the same, and a portion too long
    # for the room there is goes the other way
    options = dict(max_tokens=4096, max_slots=2, max_length=4000, max_batch_tokens=256, page_size=16)
    amply = Runner(model, device_budget_bytes=0, **options)
    tight = Runner(model, device_budget_bytes=amply.memory_plan.to_allocate() - 1, **options)
    assert tight.memory_plan.workspace < amply.memory_plan.workspace
    for runner in (amply, tight):
        calls.clear()
        compare(run_steps(runner, whole(requests)), want, "bfloat16")
        room = runner.workspace.room("latent_out", BF16)                 # (a key's latent and shared part, two heads' keys and values)
        assert len(calls) == 2 * sum(n * (48 + 64 + 2 * 128 + 2 * 128) <= room for n in (150, 64, 201))
        assert runner is tight or len(calls) == 2 * 3


@pytest.mark.parametrize("scale", [-0.1, 0.0])
def test_factors_on_the_scores_that_are_not_positive(tmp_path, monkeypatch, scale):
    """The portion kernel takes a tile's maximum before the factor, so such a layer's portions go the other way."""
    from helpers import compare, make_requests, plain_logits, portions, run_steps, whole
    from plain import pamunex_plain as P
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Runner
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 0)
    rot, mask = dict(dims=64, base=10000.0), dict(size=100)
    layers = [dict(type="latent_attention", mlp=None, mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=48, scale=scale, rot=rot, mask=mask)),
              dict(type="attention", mlp=dict(kind="dense", ff=64),
                   mixer=dict(heads=4, kv_heads=2, dim=128, vdim=128, scale=scale, rot=rot, mask=mask))]
    folder = str(tmp_path / "model")
    write_random_model(folder, config_from_dict(dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0,
                                                     layers=layers)), seed=3, matrix_std=0.12, norm_std=0.2)
    requests = make_requests(97, [150, 64, 201], seed=2)
    want, model = plain_logits(P.PlainPamunex(folder), requests), DecoderModel.load(folder, BF16)
    for cut in (whole(requests), portions(requests, (100, 65, 7))):
        runner = Runner(model, max_tokens=640, max_slots=4, max_length=256, max_batch_tokens=512, page_size=16)
        compare(run_steps(runner, cut), want, "bfloat16")


def test_made_keys_ask_for_no_plan_of_the_library(tmp_path, monkeypatch):
    """The vendor library looks a plan up for every new number of rows; of portions' keys there is another one nearly every time."""
    from helpers import make_requests
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Entry, Runner
    from mini_llm_runtime_amd.kernels import Kernels
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    latent = dict(type="latent_attention", mlp=None, mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=64, scale=192 ** -0.5,
                                                                rot=dict(dims=64, base=10000.0), mask=dict(size=4000)))
    cfg = dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=[latent])
    folder = str(tmp_path / "model")
    write_random_model(folder, config_from_dict(cfg), seed=3, matrix_std=0.12, norm_std=0.2)
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 0)
    runner = Runner(DecoderModel.load(folder, BF16), max_tokens=640, max_slots=4, max_length=512, max_batch_tokens=256, page_size=16)
    rows, made = set(), set()
    library, original = runner.kernels._lib("library_gemm"), Kernels.gemm

    def gemm(self, a, w, out, library=True):
        made.add(a.shape[0]) if not library else None
        return original(self, a, w, out, library)

    class Spied:
        def mlr_library_gemm(self, a, w, out, m, *rest):
            rows.add(m.value)
            return library.mlr_library_gemm(a, w, out, m, *rest)
    monkeypatch.setattr(Kernels, "gemm", gemm)
    monkeypatch.setitem(runner.kernels._libs, "library_gemm", Spied())
    slot, tokens = runner.open_request(), make_requests(97, [260], seed=4)["r0"]
    for lo, hi in ((0, 90), (90, 173), (173, 260)):
        runner.step([Entry(slot, tokens[lo:hi], [hi - lo - 1])])
    assert rows <= {90, 83, 87} and made == {90, 173, 260}


def test_the_page_pool_goes_before_spare_scratch_memory(tmp_path, monkeypatch):
    """A pool sized by the budget holds what it would hold without the scratch memory that made keys would like, down to a
    budget that leaves a few pages; and short portions, whose keys find room all the same, stay inside the plan."""
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Entry, MemoryBudgetError, Runner
    from mini_llm_runtime_amd.kernels import Kernels
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    latent = dict(type="latent_attention", mlp=None, mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=48, scale=192 ** -0.5,
                                                                rot=dict(dims=64, base=10000.0), mask=dict(size=4000)))
    cfg = dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=[latent, latent])
    folder = str(tmp_path / "model")
    write_random_model(folder, config_from_dict(cfg), seed=3, matrix_std=0.12, norm_std=0.2)
    model = DecoderModel.load(folder, BF16)
    runner = lambda budget: Runner(model, max_slots=3, max_length=4000, max_batch_tokens=256, page_size=16,  # noqa: E731
                                   device_budget_bytes=budget)
    ample = runner(0)
    whole = ample.memory_plan.to_allocate()
    assert ample.max_tokens >= 3 * 4000
    bare = runner(whole - 1)
    assert bare.max_tokens == ample.max_tokens and bare.memory_plan.workspace < ample.memory_plan.workspace
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 0)
    made, original = [], Kernels.portion_attention_split
    monkeypatch.setattr(Kernels, "portion_attention_split", lambda self, *a, **kw: made.append(a) or original(self, *a, **kw))
    slots = [bare.open_request(), bare.open_request()]
    bare.step([Entry(slots[0], list(range(35)), [34]), Entry(slots[1], [5], [0])])
    assert len(made) == 2 and bare.workspace.unplanned_bytes() == 0
    least = whole - ample.memory_plan.workspace - ample.memory_plan.kv_pages + bare.memory_plan.workspace      # without a page
    page = -(-ample.memory_plan.kv_pages // (ample.max_tokens // 16))
    spare = ample.memory_plan.workspace - bare.memory_plan.workspace
    for pages in (8, spare // page - 1, spare // page + 8):
        tight = runner(least + pages * page)
        assert abs(tight.max_tokens - 16 * pages) <= 16 * 2 and tight.memory_plan.workspace == bare.memory_plan.workspace
    with pytest.raises(MemoryBudgetError):
        runner(least - 1)


def test_latent_layers_of_different_windows_in_one_step(tmp_path, monkeypatch):
    """Layers of windows 1000, 30 and 1000 whose portions make their keys for other entries of a step each: the rest of the rows
    must be every layer's own, against the plain implementation."""
    from helpers import compare, make_requests, plain_logits, run_steps
    from plain import pamunex_plain as P
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Runner
    from mini_llm_runtime_amd.engine.context import StepContext
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    latent = lambda size: dict(type="latent_attention", mlp=None,  # noqa: E731
                               mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=48, scale=192 ** -0.5,
                                          rot=dict(dims=64, base=10000.0), mask=dict(size=size)))
    cfg = dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=[latent(1000), latent(30), latent(1000)])
    folder = str(tmp_path / "model")
    write_random_model(folder, config_from_dict(cfg), seed=3, matrix_std=0.12, norm_std=0.2)
    requests = make_requests(97, [250, 240, 70, 9], seed=2)
    part = lambda rid, lo, hi: dict(id=rid, tokens=requests[rid][lo:hi], want=list(range(hi - lo)))  # noqa: E731
    steps = [dict(step=0, entries=[part("r0", 0, 201), part("r3", 0, 5), part("r1", 0, 64)], end=[]),
             dict(step=1, entries=[part("r3", 5, 6), part("r0", 201, 241), part("r1", 64, 240), part("r2", 0, 50)], end=["r1"]),
             dict(step=2, entries=[part("r3", 6, 9), part("r0", 241, 250), part("r2", 50, 70)], end=["r0", "r2", "r3"])]
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 120)
    asked = []
    original = StepContext.token_groups
    monkeypatch.setattr(StepContext, "token_groups", lambda self, *a: asked.append(a[2] if len(a) > 2 else ()) or original(self, *a))
    runner = Runner(DecoderModel.load(folder, BF16), max_tokens=640, max_slots=4, max_length=256, max_batch_tokens=512, page_size=16)
    got = run_steps(runner, steps)
    assert asked[3:6] == [(1, 2), (2,), (1, 2)]                      # (the second step's three layers)
    assert runner.workspace.unplanned_bytes() == 0
    compare(got, plain_logits(P.PlainPamunex(folder), requests), "bfloat16")


def test_a_model_with_a_router_keeps_its_sums(tmp_path, monkeypatch):
    """A choice of experts turns on the last bits where two lie within rounding: prompt portions of a model that makes such
    choices keep the kernels whose order of rounding its results have always had, those of one that does not take the others."""
    from helpers import compare, make_requests, plain_logits, run_steps, whole
    from plain import pamunex_plain as P
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.engine import Runner
    from mini_llm_runtime_amd.kernels import Kernels
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.weights import write_random_model
    monkeypatch.setattr("mini_llm_runtime_amd.parts.sink_attention.PORTION_LEAST_KEYS", 0)
    calls = set()
    for name in ("portion_attention", "portion_attention_split"):
        original = getattr(Kernels, name)
        monkeypatch.setattr(Kernels, name, lambda self, *a, name=name, original=original, **kw: calls.add(name) or original(self, *a, **kw))
    requests = make_requests(97, [150, 64, 201], seed=2)
    for routed in (False, True):
        mlp = dict(kind="moe", expert=dict(ff=32), router=dict(experts=4, top=2)) if routed else dict(kind="dense", ff=64)
        layers = [dict(type="latent_attention", mlp=None, mixer=dict(heads=2, dim=128, rot_dim=64, vdim=128, kv_rank=48, scale=192 ** -0.5,
                                                                     rot=dict(dims=64, base=10000.0), mask=dict(size=100))),
                  dict(type="attention", mlp=mlp, mixer=dict(heads=4, kv_heads=2, dim=128, vdim=128, scale=128 ** -0.5,
                                                             rot=dict(dims=64, base=10000.0), mask=dict(size=100)))]
        cfg = dict(architecture="Pamunex", vocab=97, width=64, norm=dict(eps=1e-5), logit_scale=1.0, layers=layers)
        folder = str(tmp_path / f"model{routed}")
        write_random_model(folder, config_from_dict(cfg), seed=3, matrix_std=0.12, norm_std=0.2)
        runner = Runner(DecoderModel.load(folder, BF16), max_tokens=640, max_slots=4, max_length=256, max_batch_tokens=512, page_size=16)
        calls.clear()
        got = run_steps(runner, whole(requests))
        assert calls == (set() if routed else {"portion_attention", "portion_attention_split"})
        assert runner.workspace.unplanned_bytes() == 0
        if not routed:
            compare(got, plain_logits(P.PlainPamunex(folder), requests), "bfloat16")
