"""State whose two rows a slot take turns (`StateSpec(.., paired=True)`): the bookkeeping on the CPU, the kernels' two ways of naming
rows on the GPU."""
import numpy as np
import pytest
import torch


def test_a_step_that_has_run_turns_its_requests_round():
    """Sizes as planned; a step's requests change rows when it is retired and not before; the scratch request never does; a slot used
    again starts from zeros whichever row was live."""
    from mini_llm_runtime_amd.cache import CacheManager, KvSpec, StateSpec
    specs = [KvSpec(1, 16), StateSpec((6,), torch.float32, paired=True), StateSpec((3,), torch.int32), StateSpec((2, 5), torch.float32, paired=True)]
    m = CacheManager(specs, torch.float32, "cpu", page_size=8, max_tokens=64, max_slots=3, max_length=64)
    assert CacheManager.plan(specs, torch.float32, 8, 64, 3, 64) == (m.kv_bytes(), m.table_bytes(), m.state_bytes())
    assert m.has_pairs() and m.has_state() and m.state_pairs(1).shape == (8, 6) and m.state_pairs(3).shape == (8, 2, 5)
    assert m.state_view(2).shape == (4, 3) and list(m.snapshot_state()) == [2]
    slots = [m.acquire_slot() for _ in range(3)]
    everyone = np.array(slots + [m.scratch_slot])
    assert m.state_rows(everyone).tolist() == [0, 2, 4, 6] and m.state_rows([2, 2, 0]).dtype == np.int32
    for ran, rows in (([0, 2], [1, 2, 5, 6]), ([2], [1, 2, 4, 6]), ([1, 0], [0, 3, 4, 6])):
        m.prepare(ran, [1] * len(ran))
        m.commit(ran, [1] * len(ran))
        before = m.state_rows(everyone).tolist()
        m.prepare([0], [1])                                # (a step that is taken and does not run changes nothing)
        assert m.state_rows(everyone).tolist() == before
        m.retire(ran)
        assert m.state_rows(everyone).tolist() == rows
    m.state_pairs(1).fill_(7.0)
    m.release_slot(1)
    assert m.acquire_slot() == 1
    assert not m.state_pairs(1)[m.state_rows([1])].any() and m.state_pairs(1).ne(0).any(1).sum() == 7
    plain = CacheManager([StateSpec((4,))], torch.float32, "cpu", 8, 64, 2, 64)
    assert not plain.has_pairs()


@pytest.mark.gpu
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_one_slab_of_pairs_gives_what_two_slabs_give(dtype):
    """Every kernel that advances a state: outputs and written rows to the bit, rows that the step does not name untouched."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(dtype)
    gen = torch.Generator("cuda").manual_seed(3)
    heads, keys, values, offset = 2, 64, 64, 8
    lengths, slots = [40, 1, 70], [3, 0, 2]
    rows, state = sum(lengths), heads * keys * values
    ints = lambda x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    rnd = lambda *shape: torch.randn(*shape, generator=gen, device="cuda")  # noqa: E731
    q, kk, v = (rnd(rows, heads * n).to(dtype) for n in (keys, keys, values))
    decay, beta, constant = -torch.rand(rows, heads * keys, generator=gen, device="cuda"), rnd(rows, heads), -torch.rand(heads, generator=gen, device="cuda")
    first = np.concatenate([[0], np.cumsum(lengths)[:-1]]).tolist()
    cut = lambda n: [(f + i, min(n, c - i)) for f, c in zip(first, lengths) for i in range(0, c, n)]  # noqa: E731
    both = lambda pieces: (ints([f for f, _ in pieces]), ints([c for _, c in pieces]), len(pieces))  # noqa: E731
    whole = both(list(zip(first, lengths)))
    taps, bias = rnd(heads * keys, 4), rnd(heads * keys)
    positions = ints([i + (5 if n > 1 else 9) for n in lengths for i in range(n)])

    def conv(out, live, stage, where):
        y = torch.empty(rows, heads * keys, dtype=dtype, device="cuda")
        k.causal_conv(q, taps, bias, y, live, stage, offset, where, positions)
        out[:, :heads * keys] = y.float()

    def pieces(out, live, stage, where):
        some = both(cut(32))
        k.linear_recurrence(q, kk, v, decay, out, live, stage, offset, *some, where, heads, keys, values,
                            piece_state=torch.empty(some[2] * state, device="cuda"), piece_decay=torch.empty(some[2] * heads * keys, device="cuda"))

    def chunked(out, live, stage, where):
        some = both(cut(k.delta_chunk_tokens()))
        k.delta_rule_chunked(q, kk, v, decay, beta, out, live, stage, offset, *whole, where, *some,
                             torch.empty(k.delta_chunk_floats(some[2], heads, keys, values), device="cuda"), heads, keys, values)

    def decayed(out, live, stage, where):
        some = both(cut(64))
        k.decayed_recurrence_chunks(q, kk, v, constant, out, live, stage, offset, *whole, where, *some, 64,
                                    torch.empty(some[2] * state, device="cuda"), heads, keys, values)
    walks = [conv, pieces, chunked,
             lambda out, live, stage, where: k.linear_recurrence(q, kk, v, decay, out, live, stage, offset, *whole, where, heads, keys, values),
             lambda out, live, stage, where: k.delta_rule(q, kk, v, decay, beta, out, live, stage, offset, *whole, where, heads, keys, values)]
    if dtype == torch.bfloat16:
        walks.append(decayed)
    for i, walk in enumerate(walks):
        live = rnd(4, offset + state)
        stage, pairs = live.clone(), torch.full((8, offset + state), 3.0, device="cuda")
        turn = [1, 0, 0, 1]                                 # which row of slot s's pair is live
        for s in range(4):
            pairs[2 * s + turn[s]] = live[s]
        before = pairs.clone()
        got, want = torch.zeros(rows, heads * values, device="cuda"), torch.zeros(rows, heads * values, device="cuda")
        walk(want, live, stage, ints([s for s, n in zip(slots, lengths) for _ in range(n)]))
        walk(got, pairs, pairs, ints([2 * s + turn[s] for s, n in zip(slots, lengths) for _ in range(n)]))
        assert torch.equal(got, want), i
        for s in range(4):
            live_row = 2 * s + turn[s]
            assert torch.equal(pairs[live_row], before[live_row]), i
            written = pairs[live_row ^ 1]
            if s not in slots:
                assert torch.equal(written, before[live_row ^ 1]), i
            else:                                            # (what the kernel does not write of a row stays 3)
                changed = written != 3.0
                assert changed.any() and torch.equal(written[changed], stage[s][changed]) and torch.equal(stage[s][~changed], live[s][~changed]), i


@pytest.mark.gpu
def test_a_slab_that_is_only_read_need_not_come_in_pairs():
    from mini_llm_runtime_amd.kernels import KernelError, Kernels
    k = Kernels(torch.float32)
    ints = lambda *x: torch.tensor(x, dtype=torch.int32, device="cuda")  # noqa: E731
    q, decay, slab = torch.randn(1, 8, device="cuda"), -torch.rand(1, 8, device="cuda"), torch.randn(3, 64, device="cuda")
    before, outs = slab.clone(), []
    for stage in (slab, slab.clone()):
        out = torch.full((1, 8), float("nan"), device="cuda")
        k.linear_recurrence(q, q, q, decay, out, slab, stage, 0, ints(0), ints(1), 1, ints(2), 1, 8, 8, write_state=False)
        outs.append(out)
    assert torch.equal(*outs) and torch.equal(slab, before)
    with pytest.raises(KernelError, match="pairs"):
        k.linear_recurrence(q, q, q, decay, outs[0], slab, slab, 0, ints(0), ints(1), 1, ints(2), 1, 8, 8)
