"""The choice of experts, whose places the kernel counts at once, against the choice of one after the other; and the sorted pairs."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def chosen_in_rounds(scores, top, count, keep, best_alone):
    """The groups, then the experts, one after the other: the largest that is left and, among equals, the lowest index; -inf and NaN
    are never the largest, and where nothing is left the choice is expert 0."""
    per = len(scores) // count

    def largest(values):
        at, best = -1, -np.inf
        for i, v in enumerate(values):
            if v > best:
                at, best = i, v
        return at
    groups = []
    for g in range(count):
        first = second = np.float32(-np.inf)
        for v in scores[g * per:(g + 1) * per]:
            if v > first:
                first, second = v, first
            elif v > second:
                second = v
        groups.append(first + second if per >= 2 and not best_alone else first)
    left = np.full(len(scores), -np.inf, np.float32)
    for _ in range(keep):
        g = largest(groups)
        if g < 0:
            break
        groups[g] = -np.inf
        left[g * per:(g + 1) * per] = scores[g * per:(g + 1) * per]
    out = []
    for _ in range(top):
        e = largest(left)
        out.append(max(e, 0))
        left[out[-1]] = -np.inf
    return out


@pytest.mark.parametrize("best_alone", [False, True])
@pytest.mark.parametrize("rows,experts,top,count,keep", [(1, 1, 1, 1, 1), (1, 64, 64, 1, 1), (16, 20, 4, 1, 1), (17, 21, 4, 7, 2), (64, 64, 8, 8, 3), (64, 60, 5, 60, 9),
                                                         (65, 16, 4, 4, 4), (33, 65, 6, 5, 2), (40, 256, 8, 8, 4), (130, 128, 3, 1, 1),
                                                         (40, 160, 2, 8, 1), (5, 256, 1, 8, 1), (33, 128, 2, 128, 2), (900, 256, 3, 8, 2), (17, 65, 13, 5, 1)])
def test_a_place_in_the_order_is_the_choice_round_after_round(rows, experts, top, count, keep, best_alone):
    """Scores that tie in plenty, rows of infinities and NaN among them, with and without a correction; sizes of either kernel."""
    from mini_llm_runtime_amd.kernels import Kernels
    k = Kernels(torch.float32)
    rng = np.random.default_rng(rows * 1000 + experts)
    z = rng.choice(np.array([-np.inf, 0.0, 3.0, np.inf, np.nan, 1.0, -1.0], np.float32), size=(rows, experts + 1), p=[.1, .2, .1, .1, .05, .25, .2])
    z[0, :] = np.nan if rows > 1 else 0.0
    correction = rng.choice(np.array([0.0, 0.5, -np.inf], np.float32), size=experts, p=[.5, .4, .1])
    for c in (None, correction):
        ids, row_of, token_of = (torch.full(shape, -1, dtype=torch.int32, device="cuda") for shape in ((rows, top), (rows * top,), (rows * top,)))
        weights, offsets = torch.empty((rows, top), device="cuda"), torch.empty(experts + 1, dtype=torch.int32, device="cuda")
        k.router_topk(torch.from_numpy(z).cuda(), ids, weights, count, keep, correction=None if c is None else torch.from_numpy(c).cuda(),
                      renormalize=True, scale=1.5, group_score="best" if best_alone else "best_two", experts=experts)
        k.route_sort(ids, experts, offsets, token_of, row_of)
        ids_np, off, row, token = (t.cpu().numpy() for t in (ids, offsets, row_of, token_of))
        assert sorted(row.tolist()) == list(range(rows * top)) and np.array_equal(token[row], np.arange(rows * top) // top)
        assert np.array_equal(off, np.concatenate([[0], np.cumsum(np.bincount(ids_np.reshape(-1), minlength=experts))]))
        assert (off[ids_np.reshape(-1)] <= row).all() and (row < off[ids_np.reshape(-1) + 1]).all()
        with np.errstate(over="ignore"):
            scores = (1 / (1 + np.exp(-z[:, :experts]))).astype(np.float32)
        by = scores if c is None else scores + c
        assert ids_np.tolist() == [chosen_in_rounds(row, top, count, keep, best_alone) for row in by]
        plain = np.take_along_axis(scores, ids_np.astype(np.int64), 1)
        want = plain / (plain.sum(1, keepdims=True) + 1e-20) * 1.5
        np.testing.assert_allclose(weights.cpu().numpy(), want, rtol=1e-5)
