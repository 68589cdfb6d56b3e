"""The work that this engine does for its users, as cases that can be timed and compared.

A case is one model (an architecture at layer sizes of `bench.py`, random weights drawn on the GPU from the seed) and one
thing done with it over and over:

  * decode: every open request takes its next token -- one step of the batch, and the sampler's look at the logits, as a
    server's loop does it.  The requests' contexts lie between `low` and `high` tokens and grow by one a pass.
  * prompt: a request is opened, its prompt run in portions of at most 2048 tokens, the logits at its last `want` places
    returned, the request closed.  One place is what generation asks for, more are what scoring asks for.
  * mixed: one step that holds a token of every decoding request beside a whole short prompt of a new one.
  * serve: a handful of requests submitted to the scheduler and run until all are done, half of them greedy and half drawn
    at a temperature (the float32 engine, whose tokens do not hang on how a sum was rounded).

`run` returns the logits and not the tokens beside them where the engine is bfloat16: among tens of thousands of random
logits the first two often lie closer than bfloat16 rounds.  The tokens of every request's next steps are fixed beforehand
for the same reason.
"""
import math
import random

import numpy as np
import torch

PORTION = 2048                 # tokens of a prompt in one step (the scheduler's own default)
ROOM = 1024                    # tokens that a decoding request may grow by before it is filled anew

# ---- models ---------------------------------------------------------------------------------------------------------------
# layer sizes of bench.py: Qwen3 dense ...
QWEN = {
    "0.6b": dict(layers=28, hidden_size=1024, num_attention_heads=16, num_key_value_heads=8, intermediate_size=3072, tie_word_embeddings=True),
    "8b": dict(layers=36, hidden_size=4096, num_attention_heads=32, num_key_value_heads=8, intermediate_size=12288, tie_word_embeddings=False),
    "32b": dict(layers=64, hidden_size=5120, num_attention_heads=64, num_key_value_heads=8, intermediate_size=25600, tie_word_embeddings=False),
}
# ... and the two sizes that the other architectures are measured at
WIDE = {
    "2k": dict(width=2048, ff=5632, heads=16, kv=4, q_rank=768, low_rank=64, mamba_heads=64, mamba_groups=1, gla_heads=8),
    "4k": dict(width=4096, ff=12288, heads=32, kv=8, q_rank=1536, low_rank=128, mamba_heads=128, mamba_groups=8, gla_heads=16),
}
VOCAB, SPAN, KV_RANK = 32000, 1024, 512       # vocabulary, window or block of positions, latent rank of the other architectures


def _constant_decays(heads):
    return [1.0 - 2.0 ** -(2 + 6 * i / (heads - 1)) for i in range(heads)]


def _taletar(d):
    attention = dict(heads=d["heads"], kv_heads=d["kv"], dim=64, vdim=128, diff=0.6, scale=0.125, softcap=50.0,
                     q_temp=dict(coef=0.3, every=128))
    mamba = dict(heads=d["mamba_heads"], vdim=64, state=128, groups=d["mamba_groups"], conv=4, norm_groups=d["mamba_groups"])
    gla = dict(heads=d["gla_heads"], dim=128, vdim=256, rank=16, tau=16.0)
    turn = [("mamba2", mamba), ("attention", attention), ("attention", attention), ("gla", gla)]
    mlp = dict(kind="dense", ff=d["ff"], limit=7.0)
    return dict(layers=[dict(type=turn[i % 4][0], mixer=turn[i % 4][1], mlp=mlp) for i in range(8)])


def _pamunex(d):
    latent = dict(type="latent_attention", mlp=dict(kind="dense", ff=d["ff"] * 3 // 2),
                  mixer=dict(heads=d["heads"], dim=128, rot_dim=64, vdim=128, kv_rank=KV_RANK, scale=192 ** -0.5,
                             rot=dict(dims=64, base=10000.0), mask=dict(size=SPAN)))
    chunked = dict(type="attention",
                   mixer=dict(heads=d["heads"], kv_heads=d["kv"], dim=128, vdim=128, scale=128 ** -0.5,
                              rot=dict(dims=64, base=1000000.0), mask=dict(size=SPAN)),
                   mlp=dict(kind="moe", expert=dict(ff=d["ff"] * 3 // 8), router=dict(experts=8, top=2, groups=dict(count=4, keep=2))))
    return dict(logit_scale=0.5, layers=[latent if i % 2 == 0 else chunked for i in range(8)])


def _tigelorn(d):
    h, mlp = d["heads"], dict(kind="dense", ff=d["ff"])
    left = dict(heads=h, kv_heads=d["kv"], dim=128, vdim=128, scale=128 ** -0.5, rot=dict(dims=64, base=1000000.0), mask=dict(size=SPAN))
    right = dict(heads=h, dim=128, vdim=128, decay=_constant_decays(h))
    parallel = dict(type="parallel", mixer=dict(left=left, right=right, left_scale=0.5, right_scale=0.5), mlp=mlp)
    delta = dict(type="channel_delta", mlp=mlp, mixer=dict(heads=h, kv_heads=h // 2, dim=128, vdim=128, conv=4, decay_rank=d["low_rank"],
                                                          gate_rank=d["low_rank"]))
    latent = dict(type="latent_attention", mlp=mlp,
                  mixer=dict(heads=h, dim=128, rot_dim=64, vdim=128, kv_rank=KV_RANK, q_rank=d["q_rank"], scale=192 ** -0.5,
                             rot=dict(dims=64, base=10000.0, scaling=dict(factor=40.0, original=4096, fast=32.0, slow=1.0))))
    return dict(embedding=dict(bigram=dict(buckets=16381, mul_prev=1000003, mul_cur=29)), layers=[parallel, delta, latent, parallel] * 2)


def _budorax(d):
    h, mlp = d["heads"], dict(kind="moe", expert=dict(ff=d["ff"] // 2), router=dict(experts=8, top=2, scale=1.5))
    attention = dict(type="attention", mlp=mlp, mixer=dict(heads=h, kv_heads=d["kv"], dim=64, vdim=128, diff=0.6, scale=64 ** -0.5,
                                                           rot=dict(dims=64, base=1000000.0), mask=dict(size=SPAN)))
    latent = dict(type="latent_attention", mlp=mlp, mixer=dict(heads=h, dim=128, rot_dim=64, vdim=128, kv_rank=KV_RANK, q_rank=d["q_rank"],
                                                               scale=192 ** -0.5, rot=dict(dims=64, base=10000.0)))
    delta = dict(type="delta", mlp=mlp, mixer=dict(heads=h, kv_heads=h // 2, dim=128, vdim=128, conv=4))
    return dict(logit_softcap=30.0, loop=dict(start=2, stop=4, times=2), layers=[attention, latent, delta] * 2)


def _nuvorax(d):
    ff = d["ff"]
    mixer = dict(heads=d["heads"], kv_heads=d["kv"], dim=128, vdim=128, scale=128 ** -0.5, softcap=30.0,
                 rot=dict(dims=64, base=1000000.0, scaling=dict(factor=8.0, low=1.0, high=4.0, original=8192)))
    mlps = [dict(kind="dense", ff=ff * 3 // 2),
            dict(kind="moe", expert=dict(ff=ff // 4, limit=7.0), shared=dict(ff=ff // 2, limit=7.0),
                 router=dict(experts=8, top=2, scale=1.5, groups=dict(count=4, keep=2)))]
    return dict(embedding=dict(scale=8.0), logit_scale=0.5, layers=[dict(type="attention", mixer=mixer, mlp=mlps[i % 2]) for i in range(8)])


def _sagopel(d):
    h, ff, rot = d["heads"], d["ff"], dict(dims=64, base=1000000.0)
    linear = dict(heads=h, dim=128, vdim=128, decay=_constant_decays(h))
    left = dict(heads=h, kv_heads=d["kv"], dim=128, vdim=128, scale=128 ** -0.5, softcap=50.0, rot=rot, mask=dict(size=SPAN, keep_first=64))
    dense = dict(kind="dense", ff=ff)
    moe = dict(kind="moe", expert=dict(ff=ff // 8), shared=dict(ff=ff // 2), router=dict(experts=16, identity=4, top=4))
    lightning = lambda mlp: dict(type="lightning", mixer=linear, mlp=mlp)  # noqa: E731
    parallel = dict(type="parallel", mixer=dict(left=left, right=dict(linear, rot=dict(rot, dims=128))), mlp=moe)
    return dict(residual_mult=0.4, loop=dict(start=2, stop=4, times=2),
                layers=[lightning(dense), lightning(moe), parallel, lightning(moe), parallel, lightning(moe)])


FAMILIES = {"taletar": _taletar, "pamunex": _pamunex, "tigelorn": _tigelorn, "budorax": _budorax, "nuvorax": _nuvorax, "sagopel": _sagopel}


def _config(case):
    """config.json of the case's model, as a dict."""
    family, size = case["model"].split("-")
    if family == "qwen3":
        sizes = {k: v for k, v in QWEN[size].items() if k != "layers"}
        return dict(sizes, architectures=["Qwen3ForCausalLM"], head_dim=128, vocab_size=151936, max_position_embeddings=40960,
                    rms_norm_eps=1e-6, rope_theta=1000000.0, num_hidden_layers=case["layers"])
    d = WIDE[size]
    return dict(FAMILIES[family](d), architecture=family.capitalize(), vocab=VOCAB, width=d["width"], norm=dict(eps=1e-5))


def _weights(case, seed, dtype):
    """({tensor name: device tensor}, the configuration object).  Qwen3's are the random model of `bench.py`.  In the other
    architectures the token's own vector is about as large as a norm makes it and a sublayer adds a tenth of that, as in a
    trained model's stream: with every tensor from the same distribution a router's close call turns the whole row."""
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.parts import expected_tensors
    from mini_llm_runtime_amd.weights import random_tensors_on_device
    cfg = _config(case)
    parsed = config_from_dict(cfg)
    w = random_tensors_on_device(expected_tensors(parsed), seed, dtype, "cuda")
    if "architecture" in cfg:
        for name, t in w.items():
            last = name.rsplit(".", 1)[-1]
            if name in ("embed", "bigram"):
                t.mul_(0.125 / 0.02 if "scale" in cfg.get("embedding", {}) else 50.0)
            elif last == "down" or name.endswith("mix.o") or name.endswith(("left.o", "right.o")):
                t.mul_(0.2)
            elif name.endswith(("left.out", "right.out")):
                t.mul_(0.2)
            elif cfg["architecture"] == "Pamunex" and ".norm" in name and name[0] == "l" and "mix" not in name:
                t.mul_(0.1)                            # (its sublayers' outputs pass a norm before they are added)
    return w, parsed


# ---- cases ----------------------------------------------------------------------------------------------------------------
def listed():
    """Twelve cases; every kind of step, every architecture's mixers but those that a drawn case brings, both engines."""
    return [
        # one user at a terminal: the smallest step, a chain of short launches
        dict(name="decode-1", kind="decode", model="qwen3-0.6b", layers=28, dtype="bfloat16", requests=1, low=1100, high=1100),
        # the benchmark's headline: eight requests at about 4096 tokens
        dict(name="decode-8", kind="decode", model="qwen3-0.6b", layers=28, dtype="bfloat16", requests=8, low=3301, high=3907),
        # a busy server: 64 requests of all lengths on larger layers (an eighth of the model: the layers are alike)
        dict(name="decode-64", kind="decode", model="qwen3-8b", layers=4, dtype="bfloat16", requests=64, low=129, high=3001),
        # the time to a first token of an ordinary prompt
        dict(name="prompt-2000", kind="prompt", model="qwen3-0.6b", layers=28, dtype="bfloat16", tokens=2048, want=1),
        # a document: a long prompt in portions, the later ones behind many keys
        dict(name="prompt-12k", kind="prompt", model="qwen3-0.6b", layers=28, dtype="bfloat16", tokens=12321, want=1),
        # a step of a loaded server of a large model: decoded tokens beside a new prompt of odd length
        dict(name="mixed-32b", kind="mixed", model="qwen3-32b", layers=2, dtype="bfloat16", requests=32, low=200, high=2000, tokens=1501),
        # the float32 engine through the scheduler: prompts, steps of both kinds, decoding, both ways of choosing a token
        dict(name="serve-f32", kind="serve", model="qwen3-0.6b", layers=8, dtype="float32", requests=12, low=9, high=400, new=16),
        # the other architectures, each where its own mechanisms weigh most
        dict(name="taletar-decode", kind="decode", model="taletar-2k", dtype="bfloat16", requests=8, low=1000, high=1700),
        dict(name="pamunex-score", kind="prompt", model="pamunex-2k", dtype="bfloat16", tokens=1777, want=64),
        dict(name="tigelorn-prompt", kind="prompt", model="tigelorn-2k", dtype="bfloat16", tokens=2048, want=1),
        dict(name="nuvorax-mixed", kind="mixed", model="nuvorax-2k", dtype="bfloat16", requests=32, low=100, high=1500, tokens=700),
        dict(name="sagopel-decode", kind="decode", model="sagopel-2k", dtype="bfloat16", requests=48, low=100, high=1200),
    ]


def _log_uniform(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    """One more case: any model and kind of step, sizes over the whole range the listed cases span, most of them odd."""
    family = rng.choice(["qwen3", "qwen3", "qwen3"] + sorted(FAMILIES))
    if family == "qwen3":
        size = rng.choice(sorted(QWEN))
        model = dict(model=f"qwen3-{size}", layers={"0.6b": rng.randint(8, 28), "8b": rng.randint(2, 4), "32b": 2}[size])
        want, most = 1, {"0.6b": 8192, "8b": 4096, "32b": 3000}[size]
    else:
        size = rng.choice(["2k", "2k", "4k"])
        model = dict(model=f"{family}-{size}")
        want, most = 64, 2500 if size == "2k" else 1200
    kind = rng.choice(["decode", "prompt", "mixed"] + (["serve"] if family == "qwen3" and size == "0.6b" else []))
    case = dict(model, kind=kind, dtype="bfloat16")
    requests = _log_uniform(rng, 1, 64)
    low = _log_uniform(rng, 40, 900)
    high = low + _log_uniform(rng, 8, 1000 if requests > 16 else 2500)
    if kind == "decode":
        case.update(requests=requests, low=low, high=high)
    elif kind == "prompt":
        tokens = _log_uniform(rng, 17, most)
        case.update(tokens=tokens, want=min(want, tokens))
    elif kind == "mixed":
        # (few decoded rows beside a router's close call would hang on that one row)
        case.update(requests=max(requests, 24 if want > 1 else 1), low=low, high=min(high, low + 1000), tokens=_log_uniform(rng, 40, min(most, PORTION)))
    else:
        case.update(layers=rng.randint(4, 8), dtype="float32", requests=rng.randint(2, 14), low=rng.randint(3, 40), high=rng.randint(60, 400),
                    new=rng.randint(4, 16))
    if kind == "decode" and want > 1:
        case.update(requests=max(requests, 24))
    return case


def _lengths(case):
    """Tokens of every request before the pass (serve: of its prompt): from low to high, evenly over the logarithm."""
    n = case["requests"]
    return [int(round(case["low"] * (case["high"] / case["low"]) ** (i / max(1, n - 1)))) for i in range(n)]


def _vocab(case):
    return 151936 if case["model"].startswith("qwen3") else VOCAB


def _tokens(case, seed):
    """(prompts of the decoding requests, their next tokens pass by pass, the prompt of the pass)."""
    rng = np.random.default_rng(seed)
    vocab = _vocab(case)
    prompts = [rng.integers(0, vocab, n).tolist() for n in _lengths(case)] if "requests" in case else []
    after = rng.integers(0, vocab, (64, len(prompts))).tolist()
    return prompts, after, rng.integers(0, vocab, case.get("tokens", 0)).tolist()


# ---- preparing and running ------------------------------------------------------------------------------------------------
def _fill(state):
    """Opens the requests and runs their prompts, in steps of 2048 tokens that may hold parts of several."""
    from mini_llm_runtime_amd.engine import Entry
    runner = state["runner"]
    state["slots"] = slots = [runner.open_request() for _ in state["prompts"]]
    batch, free = [], PORTION
    for slot, ids in zip(slots, state["prompts"]):
        at = 0
        while at < len(ids):
            part = ids[at:at + free]
            batch.append(Entry(slot, part, []))
            at, free = at + len(part), free - len(part)
            if free == 0:
                runner.step(batch)
                batch, free = [], PORTION
    if batch:
        runner.step(batch)
    state["passes"] = 0


def prepare(case, seed):
    """A loaded model and what serves it; for decode and mixed the requests with their prompts run and the decoding steps
    captured, as a server does before its first request."""
    from mini_llm_runtime_amd.engine import Engine, EngineOptions, Runner
    from mini_llm_runtime_amd.parts import DecoderModel
    from mini_llm_runtime_amd.sampling import Sampler
    dtype = torch.bfloat16 if case["dtype"] == "bfloat16" else torch.float32
    weights, config = _weights(case, seed, dtype)
    model = DecoderModel(config, weights, dtype, "cuda:0")
    prompts, after, prompt = _tokens(case, seed)
    state = dict(case=case, prompts=prompts, after=after, prompt=prompt)
    if case["kind"] == "serve":
        state["engine"] = Engine(model, EngineOptions(max_active=8, max_model_len=1024, context_tokens=8192))
        state["seed"] = seed
        return state
    lengths = [len(p) for p in prompts]
    longest = max(lengths + [0]) + ROOM if prompts else 0
    slots = len(prompts) + (1 if prompt else 0)
    pool = sum(-(-(n + ROOM) // 64) * 64 for n in lengths) + -(-len(prompt) // 64) * 64
    rows = len(prompts) + case.get("want", 1 if prompt else 0)
    step = max(PORTION, min(len(prompt), PORTION) + len(prompts))
    state["runner"] = runner = Runner(model, max_tokens=pool, max_slots=slots, max_length=max(longest, len(prompt)), max_batch_tokens=step,
                                      max_logits_rows=rows)
    state["sampler"] = Sampler(runner.kernels, runner.device, max_rows=rows)
    state["limit"] = longest
    if case["kind"] == "decode":
        runner.warm_up(batch_sizes=[len(prompts)], contexts=[max(lengths) + 1])
    _fill(state)
    return state


def run(state):
    from mini_llm_runtime_amd.engine import Entry
    case = state["case"]
    if case["kind"] == "serve":
        engine, ids = state["engine"], []
        for i, prompt in enumerate(state["prompts"]):
            ids.append(engine.submit(prompt, max_tokens=case["new"], temperature=0.8 if i % 2 else 0.0, seed=state["seed"] + i, ignore_eos=True))
        done = engine.run_until_done()
        for i in ids:
            engine.finished.pop(i, None)
        return {"tokens": torch.tensor([done[i] for i in ids])}
    runner, sampler, prompt = state["runner"], state["sampler"], state["prompt"]
    if case["kind"] == "prompt":
        slot = runner.open_request()
        for at in range(0, len(prompt), PORTION):
            part = prompt[at:at + PORTION]
            first = max(0, len(prompt) - case["want"] - at)             # the first wanted place of this portion
            logits = runner.step([Entry(slot, part, list(range(first, len(part))))])
        runner.close_request(slot)
        return {"logits": logits}
    if runner.length(state["slots"][-1]) >= state["limit"]:             # (a program's requests end; these start over)
        for slot in state["slots"]:
            runner.close_request(slot)
        _fill(state)
    tokens = state["after"][state["passes"] % len(state["after"])]
    state["passes"] += 1
    entries = [Entry(slot, [token], [0]) for slot, token in zip(state["slots"], tokens)]
    if case["kind"] == "mixed":
        new = runner.open_request()
        logits = runner.step(entries + [Entry(new, prompt, [len(prompt) - 1])])
        runner.close_request(new)
    else:
        logits = runner.step(entries)
    zeros = [0.0] * logits.shape[0]
    sampler.sample(logits, zeros, zeros)                                # a server waits for its tokens here
    return {"logits": logits}


# ---- what a pass cannot do without ----------------------------------------------------------------------------------------
def _layers(cfg):
    """The layers in the order they run (some run twice)."""
    layers = list(range(len(cfg["layers"])))
    loop = cfg.get("loop")
    return layers if not loop else layers[:loop["start"]] + layers[loop["start"]:loop["stop"]] * loop["times"] + layers[loop["stop"]:]


def _qwen_attention(cfg):
    return dict(heads=cfg["num_attention_heads"], kv_heads=cfg["num_key_value_heads"], dim=128, vdim=128)


def _seen(kind, mixer, first, count):
    """Keys that `count` tokens from position `first` on see: (pairs of query and key, different keys)."""
    p = np.arange(first, first + count, dtype=np.int64)
    size = mixer.get("mask", {}).get("size")
    if size is None:
        start = np.zeros_like(p)
    elif kind == "block":
        start = p // size * size
    else:
        start = np.maximum(0, p - size + 1 - mixer["mask"].get("keep_first", 0))
    return int((p - start + 1).sum()), int(p[-1] - start[0] + 1)


def _mixer_work(kind, mixer, family, spans, elem):
    """(bytes, flops) of a mixer's core -- attention or recurrence, without its projections -- for spans (first, count)."""
    if kind == "parallel":
        left, right = (_mixer_work(k, mixer[k], family, spans, elem) for k in ("left", "right"))
        return left[0] + right[0], left[1] + right[1]
    h, dim, v = mixer["heads"], mixer.get("dim", mixer.get("state")), mixer["vdim"]
    tokens = sum(n for _, n in spans)
    if kind in ("mamba2", "gla", "lightning", "right", "delta", "channel_delta"):
        per = 3 if "delta" in kind else 2
        return 2 * len(spans) * h * dim * v * 4, per * 2 * tokens * h * dim * v
    seen = [_seen("block" if kind == "attention" and family in ("pamunex", "budorax") else "window", mixer, *s) for s in spans]
    pairs, keys = sum(s[0] for s in seen), sum(s[1] for s in seen)
    if kind == "latent_attention":                     # one row a token for all heads; scores and values through the latent
        return keys * (mixer["kv_rank"] + mixer["rot_dim"]) * elem, 2 * pairs * h * (2 * mixer["kv_rank"] + mixer["rot_dim"])
    maps = 2 if "diff" in mixer else 1
    flops = 2 * pairs * h * (maps * dim + maps * v) + (2 * pairs * h * h if family == "nuvorax" else 0)
    return keys * mixer["kv_heads"] * (maps * dim + v) * elem, flops


def work(case):
    """Weights read once (of a mixture the experts that the tokens choose, about), keys, values and state read once, logits
    written; the products of every token with the weights it uses, and attention or recurrence."""
    from mini_llm_runtime_amd.config import config_from_dict
    from mini_llm_runtime_amd.parts import expected_tensors
    cfg, family = _config(case), case["model"].split("-")[0]
    elem = 2 if case["dtype"] == "bfloat16" else 4
    passes = 1
    if case["kind"] == "serve":
        # (weights: once a step, of which there are about (requests / 8 slots) x new tokens)
        spans = [(0, n + case["new"] - 1) for n in _lengths(case)]
        rows, passes = case["requests"] * case["new"], -(-case["requests"] // 8) * case["new"]
    elif case["kind"] == "prompt":
        spans, rows = [(0, case["tokens"])], case["want"]
        passes = -(-case["tokens"] // PORTION)
    else:
        spans = [(n, 1) for n in _lengths(case)] + ([(0, case["tokens"])] if case["kind"] == "mixed" else [])
        rows = len(spans)
    tokens = sum(n for _, n in spans)
    head = _vocab(case) * (cfg["hidden_size"] if family == "qwen3" else cfg["width"])
    n_bytes, flops = passes * 0.0 + rows * _vocab(case) * 4 + tokens * head / _vocab(case) * elem, 2.0 * rows * head
    if family == "qwen3":
        runs = [(f"model.layers.{i}.", "attention", _qwen_attention(cfg), None) for i in range(cfg["num_hidden_layers"])]
    else:
        runs = [(f"l{i}.", cfg["layers"][i]["type"], cfg["layers"][i]["mixer"], cfg["layers"][i].get("mlp")) for i in _layers(cfg)]
    n_bytes += passes * head * elem
    sizes = {}
    for name, spec in expected_tensors(config_from_dict(cfg)).items():
        if len(spec.shape) == 2:
            sizes[name] = spec.shape[0] * spec.shape[1]
    for prefix, kind, mixer, mlp in runs:
        used = {n: s for n, s in sizes.items() if n.startswith(prefix)}
        dense = sum(s for n, s in used.items() if ".mlp.e" not in n)
        experts = sum(s for n, s in used.items() if ".mlp.e" in n)
        n_bytes += passes * dense * elem
        flops += 2.0 * tokens * dense
        if experts:
            router = mlp["router"]
            n, share = router["experts"], router["top"] / (router["experts"] + router.get("identity", 0))
            n_bytes += passes * experts * (1.0 - (1.0 - share) ** (tokens / passes)) * elem
            flops += 2.0 * tokens * share * n * (experts / n)
        b, f = _mixer_work(kind, mixer, family, spans, elem)
        n_bytes, flops = n_bytes + b, flops + f
    return {"bytes": n_bytes, "flops": flops}


def tolerance(case):
    """bfloat16: a value is rounded to 2^-9 of itself at some ten places of every layer.  Measured against 64 bits: 0.5 to
    1.4 % with Qwen3's random model, 0.2 to 0.3 % where a sublayer adds a tenth of the stream; where a mixture chooses
    otherwise on a close call, that token's row is off by some percent.  A float32 token differs where two logits or a sum
    of probabilities and the drawn number lie within 1e-6."""
    family = case["model"].split("-")[0]
    if case["kind"] == "serve":
        return {"rel": 0.0, "differ": 0.01}
    if family in ("taletar", "tigelorn"):
        return {"rel": 0.012, "max": 0.2}
    return {"rel": 0.03, "max": 0.2 if family == "qwen3" else 0.5}


# ---- the same in 64 bits --------------------------------------------------------------------------------------------------
def _f(t):
    return t.to(torch.float64)


def _linear(x, w):
    """x @ w.T in 64 bits, in blocks of rows so that the product's operands fit beside the model."""
    return x @ _f(w).T


def _rms(x, eps):
    return x / torch.sqrt((x * x).mean(-1, keepdim=True) + eps)


def _layer_norm(x, weight, bias, eps):
    d = x - x.mean(-1, keepdim=True)
    return d / torch.sqrt((d * d).mean(-1, keepdim=True) + eps) * weight + bias


def _frequencies(dims, base, scaling=None):
    """(angle a position of every pair, factor on cosine and sine) under either of the two ways to stretch them."""
    i = np.arange(dims // 2, dtype=np.float64)
    f = base ** (-2.0 * i / dims)
    if scaling is None:
        return f, 1.0
    if "fast" in scaling:
        pair = lambda turns: dims * math.log(scaling["original"] / (2.0 * math.pi * turns)) / (2.0 * math.log(base))  # noqa: E731
        lo, hi = max(math.floor(pair(scaling["fast"])), 0), min(math.ceil(pair(scaling["slow"])), dims - 1)
        ramp = np.clip((i - lo) / max(hi - lo, 0.001), 0.0, 1.0)
        return f / scaling["factor"] * ramp + f * (1.0 - ramp), 0.1 * math.log(scaling["factor"]) + 1.0
    turns = scaling["original"] * f / (2.0 * math.pi)
    blend = np.clip((turns - scaling["low"]) / (scaling["high"] - scaling["low"]), 0.0, 1.0)
    return (1.0 - blend) * f / scaling["factor"] + blend * f, 1.0


def _turn(x, rot, interleaved=False, direction=1.0):
    """x [R, T, ..., D] with the first rot["dims"] channels turned by the position t."""
    dims = rot["dims"]
    f, amp = _frequencies(dims, rot["base"], rot.get("scaling"))
    angle = direction * torch.arange(x.shape[1], dtype=torch.float64, device=x.device)[:, None] * torch.tensor(f, device=x.device)
    shape = (1, x.shape[1]) + (1,) * (x.dim() - 3) + (dims // 2,)
    c, s = (amp * torch.cos(angle)).reshape(shape), (amp * torch.sin(angle)).reshape(shape)
    out = x.clone()
    first, second = (slice(0, dims, 2), slice(1, dims, 2)) if interleaved else (slice(0, dims // 2), slice(dims // 2, dims))
    u, v = x[..., first], x[..., second]
    out[..., first], out[..., second] = u * c - v * s, v * c + u * s
    return out


def _attend(q, k, v, scale, start=None, cap=None, sink=None, keep=0, talk=None):
    """q [R, T, H, D] on keys [R, T, G, D] and values [R, T, G, V] -> [R, T, H, V].  `start`: the first key that the query at
    each position sees (and the first `keep` besides); `sink` [H]: one more summand exp(sink) of the softmax; `talk` [H, H]
    mixes the heads' weights before they meet the values."""
    R, T, H, _ = q.shape
    g = H // k.shape[2]
    spread = lambda t: t.permute(0, 2, 1, 3).repeat_interleave(H // t.shape[2], 1) if g > 1 else t.permute(0, 2, 1, 3)  # noqa: E731
    kh, vh = spread(k).transpose(2, 3).contiguous(), spread(v).contiguous()
    out = torch.empty(R, T, H, v.shape[3], dtype=torch.float64, device=q.device)
    step = max(16, min(T, int(1.5e8 / (R * H * T))))
    j = torch.arange(T, device=q.device)
    for at in range(0, T, step):
        end = min(T, at + step)
        s = (q[:, at:end].permute(0, 2, 1, 3).contiguous() @ kh[..., :end]) * scale
        if cap is not None:
            s = cap * torch.tanh(s / cap)
        p = j[at:end, None]
        seen = j[None, :end] <= p
        if start is not None:
            seen = seen & ((j[None, :end] >= start[at:end, None]) | (j[None, :end] < keep))
        s = s.masked_fill(~seen, -math.inf)
        top = s.amax(-1, keepdim=True)
        if sink is not None:
            sk = sink.reshape(1, H, 1, 1)
            top = torch.maximum(top, sk)
        e = torch.exp(s - top)
        total = e.sum(-1, keepdim=True)
        if sink is not None:
            total = total + torch.exp(sk - top)
        e = e / total
        if talk is not None:
            e = (talk @ e.reshape(R, H, -1)).reshape(e.shape)
        out[:, at:end] = (e @ vh[:, :, :end]).permute(0, 2, 1, 3)
    return out


def _starts(kind, size, T, device):
    p = torch.arange(T, device=device)
    return None if size is None else p // size * size if kind == "block" else (p - size + 1).clamp(min=0)


def _recur(q, k, v, decay, beta=None):
    """S <- decay S + k v^T (with `beta` the delta rule: k (beta (v - S^T k))^T), o = S^T q.  q, k, decay [R, T, H, N] (decay's
    last axis may be 1), v [R, T, H, V]."""
    R, T, H, N = k.shape
    S = torch.zeros(R, H, N, v.shape[3], dtype=torch.float64, device=k.device)
    out = torch.empty(R, T, H, v.shape[3], dtype=torch.float64, device=k.device)
    for t in range(T):
        kt, vt = k[:, t, :, :, None], v[:, t, :, None, :]
        S = S * decay[:, t, :, :, None]
        if beta is not None:
            vt = beta[:, t, :, None, None] * (vt - (S * kt).sum(2, keepdim=True))
        S = torch.addcmul(S, kt, vt)
        out[:, t] = (q[:, t, :, None, :] @ S)[:, :, 0]
    return out


def _conv(x, taps, bias=0.0):
    T, n = x.shape[1], taps.shape[1]
    y = torch.zeros_like(x) + bias
    for j in range(min(n, T)):
        y[:, j:] += x[:, :T - j] * taps[:, n - 1 - j]
    return y


silu = torch.nn.functional.silu
softplus = torch.nn.functional.softplus


def _diff_attention(x, w, m, eps, family):
    R, T, _ = x.shape
    H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k = _linear(x, w["q"]).reshape(R, T, H, 2, D), _linear(x, w["k"]).reshape(R, T, G, 2, D)
    v = _linear(x, w["v"]).reshape(R, T, G, V)
    if "q_temp" in m:
        p = torch.arange(T, dtype=torch.float64, device=x.device)
        q = q * (1.0 + m["q_temp"]["coef"] * torch.log(torch.floor((p + 1) / m["q_temp"]["every"]) + 1.0)).reshape(1, T, 1, 1, 1)
    if "rot" in m:
        q, k = _turn(q, m["rot"], True), _turn(k, m["rot"], True)
    lam = torch.exp((_f(w["lq1"]) * _f(w["lk1"])).sum()) - torch.exp((_f(w["lq2"]) * _f(w["lk2"])).sum()) + m["diff"]
    start = _starts("block", m.get("mask", {}).get("size"), T, x.device)
    maps = [_attend(q[:, :, :, i], k[:, :, :, i], v, m["scale"], start, m.get("softcap")) for i in (0, 1)]
    o = (_rms(maps[0] - lam * maps[1], eps) * (1.0 - m["diff"])).reshape(R, T, H * V)
    return _linear(o * torch.sigmoid(_linear(x, w["g"])) if "g" in w else o, w["o"])


def _plain_attention(x, w, m, eps, family):
    """Grouped-query attention of Qwen3, Pamunex (blocks of positions, a sink), Tigelorn and Sagopel (windows) and Nuvorax
    (turned values, mixed heads)."""
    R, T, _ = x.shape
    H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    part = lambda n, h, d: (_linear(x, w[n]) + (_f(w[n + ".b"]) if n + ".b" in w else 0.0)).reshape(R, T, h, d)  # noqa: E731
    q, k, v = part("q", H, D), part("k", G, D), part("v", G, V)
    if "q.norm" in w:
        q, k = _rms(q, eps) * _f(w["q.norm"]), _rms(k, eps) * _f(w["k.norm"])
    q, k = _turn(q, m["rot"]), _turn(k, m["rot"])
    if family == "tigelorn":
        q, k = _rms(q, eps), _rms(k, eps)
    mask = m.get("mask", {})
    start = _starts("block" if family == "pamunex" else "window", mask.get("size"), T, x.device)
    sink = _f(w["sink"]) if "sink" in w else torch.zeros(H, dtype=torch.float64, device=x.device) if family == "nuvorax" else None
    values = dict(dims=V, base=m["rot"]["base"])
    o = _attend(q, k, _turn(v, values) if family == "nuvorax" else v, m["scale"], start, m.get("softcap"), sink, mask.get("keep_first", 0),
                _f(w["talk"]) if "talk" in w else None)
    if family == "nuvorax":
        o = _turn(o, values, direction=-1.0) * torch.sigmoid(_linear(x, w["g"]))[..., None]
    o = o.reshape(R, T, H * V)
    return _linear(o * torch.sigmoid(_linear(x, w["g"])) if family == "tigelorn" else o, w["o"])


def _latent_attention(x, w, m, eps, family):
    R, T, _ = x.shape
    H, D, C, V = m["heads"], m["dim"], m["kv_rank"], m["vdim"]
    pairs = family != "pamunex"                        # (neighbouring channels, or channels half a part away)
    q = _linear(_rms(_linear(x, w["dq"]), eps) * _f(w["dq.norm"]), w["uq"]) if "dq" in w else _linear(x, w["q"])
    q = q.reshape(R, T, H, -1)
    down = _linear(x, w["dkv"])
    latent = _rms(down[..., :C], eps) * _f(w["dkv.norm"])
    k_turned = _turn(down[..., None, C:], m["rot"], pairs).expand(R, T, H, m["rot_dim"])
    k = torch.cat([_linear(latent, w["uk"]).reshape(R, T, H, D), k_turned], -1)
    q = torch.cat([q[..., :D], _turn(q[..., D:], m["rot"], pairs)], -1)
    start = _starts("window", m.get("mask", {}).get("size"), T, x.device)
    o = _attend(q, k, _linear(latent, w["uv"]).reshape(R, T, H, V), m["scale"], start, None, _f(w["sink"]) if "sink" in w else None)
    if "g" in w:
        o = o * torch.sigmoid(_linear(x, w["g"]))[..., None]
    return _linear(o.reshape(R, T, H * V), w["o"])


def _constant_decay(x, w, m, eps, family, turned=False):
    """Linear attention with a constant decay a head; `turned`: retention, whose queries and keys are turned instead."""
    R, T, _ = x.shape
    H, D, V = m["heads"], m["dim"], m["vdim"]
    act = (lambda t: t) if turned else silu
    q, k, v = (act(_linear(x, w[n])).reshape(R, T, H, -1) for n in "qkv")
    if turned:
        q, k = _turn(q, m["rot"]), _turn(k, m["rot"]) * D ** -0.5
    decay = torch.tensor(m["decay"], dtype=torch.float64, device=x.device).reshape(1, 1, H, 1).expand(R, T, H, 1)
    o = _recur(q, k, v, decay)
    gate = _linear(x, w["g"])
    o = _rms(o, eps).reshape(R, T, H * V) * silu(gate) if turned else _rms(o.reshape(R, T, H * V), eps) * _f(w["norm"]) * torch.sigmoid(gate)
    return _linear(o, w["o"])


def _gla(x, w, m, eps, family):
    R, T, _ = x.shape
    H, D, V = m["heads"], m["dim"], m["vdim"]
    q, k, v = (_linear(x, w[n]).reshape(R, T, H, -1) for n in "qkv")
    decay = torch.sigmoid(_linear(_linear(x, w["a1"]), w["a2"]) + _f(w["a2.b"])) ** (1.0 / m["tau"])
    o = _rms(_recur(q * D ** -0.5, k, v, decay.reshape(R, T, H, D)), eps) * _f(w["norm"])
    return _linear(o.reshape(R, T, H * V) * silu(_linear(x, w["g"])), w["o"])


def _mamba2(x, w, m, eps, family):
    R, T, _ = x.shape
    H, V, N, G = m["heads"], m["vdim"], m["state"], m["groups"]
    inner = H * V
    p = _linear(x, w["in"])
    z, dt = p[..., :inner], softplus(p[..., 2 * inner + 2 * G * N:] + _f(w["dt_bias"]))
    xbc = silu(_conv(p[..., inner:2 * inner + 2 * G * N], _f(w["conv"]), _f(w["conv.b"])))
    u = xbc[..., :inner].reshape(R, T, H, V)
    B, C = (xbc[..., inner + i * G * N:inner + (i + 1) * G * N].reshape(R, T, G, N).repeat_interleave(H // G, 2) for i in (0, 1))
    y = _recur(C, B, dt[..., None] * u, torch.exp(-torch.exp(_f(w["A_log"])) * dt)[..., None]) + _f(w["D"])[:, None] * u
    y = (y.reshape(R, T, inner) * silu(z)).reshape(R, T, m["norm_groups"], -1)
    return _linear(_rms(y, eps).reshape(R, T, inner) * _f(w["norm"]), w["o"])


def _delta(x, w, m, eps, family):
    R, T, _ = x.shape
    H, G, D, V = m["heads"], m["kv_heads"], m["dim"], m["vdim"]
    q, k, v = (silu(_conv(_linear(x, w[n]), _f(w[n + ".conv"]))) for n in "qkv")
    unit = lambda t: (t / torch.sqrt((t * t).sum(-1, keepdim=True) + 1e-6)).repeat_interleave(H // G, 2)  # noqa: E731
    q, k, v = unit(q.reshape(R, T, G, D)) * D ** -0.5, unit(k.reshape(R, T, G, D)), v.reshape(R, T, H, V)
    rate = _linear(_linear(x, w["a1"]), w["a2"]) if "a1" in w else _linear(x, w["a"])
    rate = softplus(rate + _f(w["dt_bias"])).reshape(R, T, H, -1)
    decay = torch.exp(-torch.exp(_f(w["A_log"])).reshape(1, 1, H, 1) * rate)
    gate = torch.sigmoid(_linear(_linear(x, w["g1"]), w["g2"])) if "g1" in w else silu(_linear(x, w["g"]))
    o = _rms(_recur(q, k, v, decay, torch.sigmoid(_linear(x, w["b"]))), eps) * _f(w["norm"]) * gate.reshape(R, T, H, V)
    return _linear(o.reshape(R, T, H * V), w["o"])


def _sub(w, prefix):
    return {n[len(prefix):]: t for n, t in w.items() if n.startswith(prefix)}


def _both(x, w, m, eps, family):
    left = _plain_attention(x, _sub(w, "left."), m["left"], eps, family)
    right = _constant_decay(x, _sub(w, "right."), m["right"], eps, family, turned=family == "sagopel")
    if family == "tigelorn":
        return m["left_scale"] * left + m["right_scale"] * right
    return 0.5 * (_rms(left, eps) * _f(w["left.out"]) + _rms(right, eps) * _f(w["right.out"]))


def _mixer(kind, family):
    return {"attention": _diff_attention if family in ("taletar", "budorax") else _plain_attention, "latent_attention": _latent_attention,
            "lightning": _constant_decay, "parallel": _both, "gla": _gla, "mamba2": _mamba2, "delta": _delta, "channel_delta": _delta}[kind]


def _glu(x, w, act, limit=None):
    out = []
    gate, up, down = _f(w["gate"]).T, _f(w["up"]).T, _f(w["down"]).T
    for rows in x.reshape(-1, x.shape[-1]).split(4096):
        g, u = rows @ gate, rows @ up
        if limit is not None:
            g, u = g.clamp(max=limit), u.clamp(-limit, limit)
            out.append((g * torch.sigmoid(1.702 * g) * (u + 1.0)) @ down)
        else:
            out.append((act(g) * u) @ down)
    return torch.cat(out).reshape(x.shape)


def _two_matrices(x, w, act):
    return torch.cat([act(_linear(rows, w["up"])) @ _f(w["down"]).T for rows in x.reshape(-1, x.shape[-1]).split(4096)]).reshape(x.shape)


def _choose(x, w, mlp, family):
    """(experts [N, top], their weights): every architecture's way to choose, the lower number on a tie."""
    r = mlp["router"]
    z = _linear(x, w["router"])
    s = torch.sigmoid(z) if family in ("pamunex", "budorax") else torch.softmax(z, -1)
    choice = s + _f(w["correction"]) if "correction" in w else s
    if "groups" in r:
        blocks = s.reshape(s.shape[0], r["groups"]["count"], -1)
        score = blocks.topk(2, -1)[0].sum(-1) if family == "pamunex" else blocks.amax(-1)
        keep = torch.zeros_like(score, dtype=torch.bool).scatter_(1, score.topk(r["groups"]["keep"], -1)[1], True)
        choice = choice.masked_fill(~keep.repeat_interleave(blocks.shape[2], 1), -math.inf)
    ids = choice.topk(r["top"], -1)[1]
    picked = s.gather(1, ids)
    return ids, picked / (picked.sum(-1, keepdim=True) + 1e-20) * r["scale"] if "scale" in r else picked


def _feed_forward(x, w, mlp, family):
    relu2 = lambda t: torch.relu(t) ** 2  # noqa: E731
    gelu = lambda t: torch.nn.functional.gelu(t, approximate="tanh")  # noqa: E731
    one = {"pamunex": lambda t, u: _two_matrices(t, u, relu2), "budorax": lambda t, u: _glu(t, u, silu),
           "nuvorax": lambda t, u: _glu(t, u, None, mlp["expert"]["limit"]), "sagopel": lambda t, u: _glu(t, u, silu)}.get(family)
    if mlp["kind"] == "dense":
        return {"taletar": lambda: _glu(x, w, None, mlp.get("limit")), "tigelorn": lambda: _glu(x, w, gelu), "pamunex": lambda: one(x, w),
                "nuvorax": lambda: _two_matrices(x, w, torch.nn.functional.gelu), "sagopel": lambda: _glu(x, w, torch.relu),
                "qwen3": lambda: _glu(x, w, silu)}[family]()
    rows = x.reshape(-1, x.shape[-1])
    ids, weights = _choose(rows, w, mlp, family)
    out = torch.zeros_like(rows)
    n = mlp["router"]["experts"]
    for e in range(n):
        at, which = torch.nonzero(ids == e, as_tuple=True)
        if at.numel():
            out.index_add_(0, at, weights[at, which][:, None] * one(rows[at], _sub(w, f"e{e}.")))
    if "identity" in mlp["router"]:
        out += (weights * (ids >= n)).sum(-1, keepdim=True) * rows
    if "shared.gate" in w:
        y = one(rows, _sub(w, "shared."))
        out += y * torch.sigmoid(_linear(rows, w["shared.sg"])) if "shared.sg" in w else y
    return out.reshape(x.shape)


def _qwen_names(w):
    """The tensors of a Qwen3 model under the names that the functions here use."""
    short = {"input_layernorm.weight": "norm1", "post_attention_layernorm.weight": "norm2", "self_attn.q_norm.weight": "mix.q.norm",
             "self_attn.k_norm.weight": "mix.k.norm"}
    out = {"embed": w["model.embed_tokens.weight"], "final.norm": w["model.norm.weight"]}
    out["head"] = w.get("lm_head.weight", out["embed"])
    for name, t in w.items():
        if name.startswith("model.layers."):
            layer, rest = name[len("model.layers."):].split(".", 1)
            out[f"l{layer}." + short.get(rest, rest.replace("self_attn.", "mix.").replace("_proj.weight", ""))] = t
    return out


def _hidden_logits(cfg, w, family, ids, want):
    """Logits [R, len(want row), vocab] of sequences ids [R, T] (those shorter than T are filled up behind) at places want [R, n]."""
    eps = cfg["rms_norm_eps"] if family == "qwen3" else cfg["norm"]["eps"]
    if family == "qwen3":
        layers = [dict(type="attention", mixer=dict(_qwen_attention(cfg), scale=128 ** -0.5, rot=dict(dims=128, base=cfg["rope_theta"])),
                       mlp=dict(kind="dense"))] * cfg["num_hidden_layers"]
        order = range(len(layers))
    else:
        layers, order = cfg["layers"], _layers(cfg)
    x = _f(w["embed"][ids]) * cfg.get("embedding", {}).get("scale", 1.0)
    if family == "tigelorn":
        b = cfg["embedding"]["bigram"]
        rows = torch.full_like(ids, b["buckets"])
        rows[:, 1:] = (ids[:, :-1] * b["mul_prev"] + ids[:, 1:] * b["mul_cur"]) % b["buckets"]
        x = x + _f(w["bigram"][rows])
    x0 = x
    around = 1.0 if family == "tigelorn" else 0.0

    def norm(name, t):
        if family == "budorax":
            return torch.tanh(_f(w[name + ".alpha"]) * t) * _f(w[name]) + _f(w[name + ".b"])
        if family in ("pamunex", "nuvorax"):
            return _layer_norm(t, _f(w[name]), _f(w[name + ".b"]) if name + ".b" in w else 0.0, eps)
        return _rms(t, eps) * (_f(w[name]) + around)
    passes = 0
    for i in order:
        layer, name = layers[i], f"l{i}."
        if cfg.get("loop") and i == cfg["loop"]["start"]:
            if family == "sagopel":
                x = x + _f(w["loop.step"][passes])
            elif passes:
                x = x + x0
            passes += 1
        mix, mlp = _sub(w, name + "mix."), _sub(w, name + "mlp.")
        mixer = lambda t: _mixer(layer["type"], family)(t, mix, layer["mixer"], eps, family)  # noqa: B023,E731
        feed = lambda t: _feed_forward(t, mlp, layer["mlp"], family)  # noqa: B023,E731
        if family == "pamunex":
            x = x + norm(name + "norm1", mixer(x))
            x = x + norm(name + "norm2", feed(x))
        elif family == "budorax":
            x = x + norm(name + "norm1b", mixer(norm(name + "norm1", x)))
            x = x + norm(name + "norm2b", feed(norm(name + "norm2", x)))
        elif family == "nuvorax":
            h = norm(name + "norm1", x)
            x = x + mixer(h) + feed(h)
        elif family == "taletar":                      # (both sublayers read the stream before either)
            x = x + mixer(norm(name + "norm1", x)) + feed(norm(name + "norm2", x))
        else:
            m = cfg.get("residual_mult", 1.0)
            x = x + m * mixer(norm(name + "norm1", x))
            x = x + m * feed(norm(name + "norm2", x))
    x = norm("final.norm", x.gather(1, want[:, :, None].expand(-1, -1, x.shape[2])))
    logits = _linear(x, w.get("head", w["embed"])) * cfg.get("logit_scale", 1.0)
    cap = cfg.get("logit_softcap")
    return logits if cap is None else cap * torch.tanh(logits / cap)


def exact(case, seed):
    """The first pass's logits in 64 bits, on the GPU, from whole sequences and without a cache; nothing where only tokens come
    back (serve) or where it would take too long."""
    if case["kind"] == "serve" or work(dict(case, kind="prompt", tokens=sum(_lengths(case)) if "requests" in case else case["tokens"],
                                            want=1))["flops"] > 3e14:
        return None
    cfg, family = _config(case), case["model"].split("-")[0]
    w = _weights(case, seed, torch.bfloat16)[0]
    w = _qwen_names(w) if family == "qwen3" else w
    prompts, after, prompt = _tokens(case, seed)
    whole = [p + [t] for p, t in zip(prompts, after[0])]
    with torch.no_grad():
        rows, at = [], 0
        while at < len(whole):                         # sequences of similar length together, at most 16384 places
            n = 1
            while at + n < len(whole) and (n + 1) * len(whole[at + n]) <= 16384:
                n += 1
            part = whole[at:at + n]
            longest = max(len(p) for p in part)
            ids = torch.tensor([p + [0] * (longest - len(p)) for p in part], device="cuda")
            want = torch.tensor([[len(p) - 1] for p in part], device="cuda")
            rows.append(_hidden_logits(cfg, w, family, ids, want)[:, 0])
            at += n
        if prompt:
            first = len(prompt) - case.get("want", 1)
            want = torch.arange(first, len(prompt), device="cuda")[None]
            rows.append(_hidden_logits(cfg, w, family, torch.tensor([prompt], device="cuda"), want)[0])
        return {"logits": torch.cat(rows)}


if __name__ == "__main__":
    for one in listed() + [draw(random.Random(i)) for i in range(6)]:
        print(one, work(one), tolerance(one))
