"""A step's inputs: the native pass over a batch's entries, the vectors for the device, and the block tables' way there."""
import ctypes

import numpy as np
import pytest
import torch

from mini_llm_runtime_amd.engine import Entry
from mini_llm_runtime_amd.kernels import build

VOCAB, TOKENS, ROWS = 1000, 64, 12


def gathered(entries, vocab=VOCAB):
    """What the native pass makes of the entries, or None where it leaves them to the caller."""
    ids, counts, slots, places, rows, totals = (np.full(max(n, 1), -7, np.int32) for n in (TOKENS, TOKENS, TOKENS, TOKENS, ROWS, 4))
    rc = build.load("step_inputs").mlr_step_entries(ctypes.py_object(entries), ctypes.c_long(vocab), TOKENS, ROWS,
                                                    *(ctypes.c_void_p(v.ctypes.data) for v in (ids, counts, slots, places, rows, totals)))
    assert rc in (0, 1)
    if rc:
        return None
    n, total, r, single = totals.tolist()
    return ids[:total].tolist(), counts[:n].tolist(), slots[:n].tolist(), places[:n].tolist(), rows[:r].tolist(), bool(single)


@pytest.mark.parametrize("batch,single", [
    ([(3, [5], [0])], True), ([(0, [0], [0]), (7, [VOCAB - 1], [0])], True), ([(1, (4, 5, 6), (0, 2)), (2, [9], [])], False),
    ([(1, [1] * TOKENS, list(range(ROWS)))], False), ([(4, [8], [])], False), ([(i, [i], [0]) for i in range(ROWS)], True)])
def test_a_plain_batch_is_read_in_one_pass(batch, single):
    entries = [Entry(*e) for e in batch]
    starts = np.cumsum([0] + [len(e.tokens) for e in entries])
    assert gathered(entries) == ([t for e in entries for t in e.tokens], [len(e.tokens) for e in entries], [e.slot for e in entries],
                                 [len(e.want) for e in entries], [int(s) + w for s, e in zip(starts, entries) for w in e.want], single)


@pytest.mark.parametrize("entries", [
    [], (Entry(0, [1], []),), [Entry(0, [], [])], [Entry(0, [VOCAB], [])], [Entry(0, [-1], [])], [Entry(0, [1 << 70], [])], [Entry(0, [1.0], [])],
    [Entry(0, [True], [])], [Entry(0, np.array([1, 2]), [])], [Entry(0, ["1"], [])], [Entry(0, [1], [1])], [Entry(0, [1], [-1])],
    [Entry(0, [1, 2], [1, 0])], [Entry(0, [1, 2], [1, 1])], [Entry(0, [1], range(1))], [Entry(-1, [1], [0])], [Entry(None, [1], [0])],
    [Entry(0, [1] * (TOKENS + 1), [])], [Entry(0, [1] * 40, list(range(ROWS + 1)))], [object()], [Entry(0, [1] * 40, []), Entry(1, [1] * 25, [])],
    [Entry(np.int64(0), [1], [0])], [Entry(0, None, [])]])
def test_any_other_batch_is_left_to_the_caller(entries):
    """Refusals with their messages, and the forms that are taken element by element (numpy vectors, places in any order)."""
    assert gathered(entries) is None


def test_entries_that_are_more_than_tuples_of_values():
    """Attributes that are code: one that raises, one that empties the list it is read from."""
    class Odd:
        want, tokens = [0], [3]

        def __init__(self, act):
            self.act = act

        @property
        def slot(self):
            return self.act()

    def fails():
        raise RuntimeError("no slot")
    assert gathered([Odd(fails)]) is None
    entries = []
    entries += [Odd(lambda: (entries.clear(), 5)[1]), Odd(lambda: 6)]
    assert gathered(entries) == ([3], [1], [5], [1], [0], True)


@pytest.mark.parametrize("tokens", [b"\x05", bytearray(b"\x03\x04"), {7}, {9: "a"}, range(3), np.array([5, 6]), [np.int64(4)], (True,), [4.0], torch.tensor([8, 2]),
                                    b"\x01" * 17, range(20)])
def test_odd_forms_of_tokens_become_the_same_batch(tokens):
    """What the native pass leaves to the Python one is taken as any list of the same numbers is."""
    from types import SimpleNamespace
    from mini_llm_runtime_amd.engine.step import Runner
    r = object.__new__(Runner)
    r.poisoned, r.max_batch_tokens, r.max_logits_rows, r.model = False, TOKENS, ROWS, SimpleNamespace(spec=SimpleNamespace(vocab_size=VOCAB))
    ids, counts, slots, places, rows, totals = (np.full(n, -7, np.int32) for n in (TOKENS, TOKENS, TOKENS, TOKENS, ROWS, 4))
    r._plain, r._plain_at, r._inputs = [ids, counts, slots, places, np.empty(TOKENS, np.int32), rows, totals], None, build.load("step_inputs")
    r._plain_args = (ctypes.c_long(VOCAB), TOKENS, ROWS, *(ctypes.c_void_p(v.ctypes.data) for v in (ids, counts, slots, places, rows, totals)))
    numbers = [int(t) for t in tokens]
    def made(batch):
        assert len(batch.first) == len(batch.slots) and batch.ids.dtype == np.int32
        return [v.tolist() for v in (batch.ids, batch.counts, batch.slots, batch.want_rows)] + [batch.total, batch.single]
    for first in ([Entry(1, [3, 4], [1])], [], [Entry(3, [8], [0])]):
        want = made(r._gather([*first, Entry(2, numbers, [0])]))
        assert made(r._gather([*first, Entry(2, tokens, [0])])) == want
        assert made(r._gather([*first, Entry(np.int64(2), numbers, np.array([0]))])) == want


def test_without_the_interpreters_headers_every_batch_is_read_entry_by_entry(tmp_path, monkeypatch):
    """The library that reads Python objects cannot be compiled there (and says what is missing); all others are."""
    made = []
    monkeypatch.setattr(build, "_python_include", lambda: str(tmp_path))
    monkeypatch.setattr(build, "_lib_dir", lambda: str(tmp_path))
    monkeypatch.setattr(build, "_compile", lambda out, cmd, digest: made.append(out))
    assert not build.available("step_inputs") and build.available("host")
    with pytest.raises(build.BuildError, match="Python.h"):
        build.ensure_built(["step_inputs"], verbose=False)
    build.build_all(verbose=False)
    assert len(made) == len(build.HOST_LIBRARIES) - 1 + sum(2 if v[2] else 1 for v in build.HIP_LIBRARIES.values())
    assert not any("step_inputs" in out for out in made)
    out, _, digest = build._plan("step_inputs", None)
    (tmp_path / "Python.h").touch()
    assert build.available("step_inputs")
    (tmp_path / "Python.h").unlink()
    with open(out, "w"), open(out + ".stamp", "w") as stamp:
        stamp.write(digest)
    assert build.available("step_inputs")                   # (built elsewhere)


@pytest.mark.gpu
def test_a_runner_without_the_native_pass(model_folders, monkeypatch):
    """The same logits to the bit: whole prompts, portions beside single tokens, captured steps with rows of the scratch request."""
    from conftest import PAGE_SIZE, TINY
    from helpers import last_one_by_one, make_requests, mixed, run_steps, whole
    from mini_llm_runtime_amd.engine import Runner
    from mini_llm_runtime_amd.parts import DecoderModel
    model = DecoderModel.load(model_folders["A"], torch.float32)
    reqs = make_requests(TINY["A"]["vocab_size"], [40, 13, 70, 2, 29], seed=3)
    got = []
    for there in (True, False):
        monkeypatch.setattr(build, "available", lambda name: there or name != "step_inputs")
        r = Runner(model, max_tokens=640, max_slots=6, max_length=160, max_batch_tokens=160, page_size=PAGE_SIZE["A"])
        assert (r._inputs is not None) == there
        got.append([run_steps(r, steps) for steps in (whole(reqs), mixed(reqs, seed=2)[0], last_one_by_one(reqs, tail=8))])
    for with_it, without in zip(*got):
        assert with_it.keys() == without.keys()
        for i in with_it:
            assert np.array_equal(with_it[i], without[i], equal_nan=True)


@pytest.mark.parametrize("fill,fill_first", [(0, False), (3, False), (2, True)])
def test_the_rows_of_a_step(fill, fill_first):
    counts, slots, first = (np.array(v, np.int32) for v in ([1, 4, 2], [5, 0, 9], [17, 0, 300]))
    ids = np.arange(100, 107, dtype=np.int32)
    out = np.full((3, 7 + fill), -1, np.int32)
    build.load("step_inputs").mlr_step_rows(3, 7, *(ctypes.c_void_p(v.ctypes.data) for v in (ids, counts, slots, first)), fill, int(fill_first), 11,
                                            ctypes.c_void_p(out.ctypes.data))
    rows = [ids.tolist(), [17, 0, 1, 2, 3, 300, 301], [5, 0, 0, 0, 0, 9, 9]]
    extra = [[0] * fill, [0] * fill, [11] * fill]
    assert out.tolist() == [e + r if fill_first else r + e for r, e in zip(rows, extra)]


@pytest.mark.gpu
@pytest.mark.parametrize("slots,length", [(40, 40960), (40, 512), (1, 128)])
def test_changed_rows_of_the_block_tables_reach_the_device(slots, length):
    """Rows far apart in a large table go one by one, in a small one as one piece with what lies between."""
    from mini_llm_runtime_amd.cache.manager import CacheManager, KvSpec
    cache = CacheManager([KvSpec(1, 16)], torch.float32, torch.device("cuda:0"), 16, 4096, slots, length)
    for _ in range(slots):
        cache.acquire_slot()
    table = cache._tables[0]
    for step in ([0, slots - 1], [slots // 2], list(range(0, slots, 3)), [slots - 1]):
        step = sorted(set(step))
        first = np.full(len(step), -1, np.int32)
        lengths = [cache.length(s) for s in step]
        cache.commit_into(np.array(step, np.int32), np.full(len(step), 17, np.int32), first)
        assert first.tolist() == lengths
        assert np.array_equal(table[:slots].cpu().numpy(), cache.book.table(0))
