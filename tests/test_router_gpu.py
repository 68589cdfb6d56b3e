"""The router's product and choice in one launch: the logits against 64 bits, the choice that of the kernel that takes logits, bit by
bit, and the sizes that go the other way."""
import pytest
import torch

from mini_llm_runtime_amd.kernels import Kernels

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,width,outputs,experts,top,groups,score", [
    (1, 8, 1, 1, 1, (1, 1, "best"), "sigmoid"), (3, 72, 5, 4, 2, (2, 1, "best_two"), "softmax"), (48, 2048, 20, 20, 4, (1, 1, "best"), "softmax"),
    (33, 520, 65, 64, 8, (8, 4, "best_two"), "sigmoid"), (7, 4096, 9, 8, 2, (4, 2, "best"), "softmax"), (1777, 2048, 8, 8, 2, (4, 2, "best_two"), "sigmoid"),
    (2100, 2048, 8, 8, 2, (1, 1, "best"), "sigmoid"), (4, 512, 80, 80, 3, (1, 1, "best"), "softmax"), (5, 100, 6, 6, 2, (1, 1, "best"), "sigmoid")])
def test_router_in_one_launch(rows, width, outputs, experts, top, groups, score):
    gen = torch.Generator().manual_seed(3)
    k = Kernels(torch.bfloat16)
    x, w = torch.randn((rows, width), generator=gen).bfloat16().cuda(), (torch.randn((outputs, width), generator=gen) * 0.05).bfloat16().cuda()
    correction = torch.randn(experts, generator=gen).cuda() * 0.1
    made = lambda: (torch.full((rows, outputs), float("nan"), device="cuda"), torch.full((rows, top), -1, dtype=torch.int32, device="cuda"),  # noqa: E731
                    torch.full((rows, top), float("nan"), device="cuda"))
    z, ids, weights = made()
    how = dict(correction=correction, renormalize=True, scale=1.5, score=score, group_score=groups[2], experts=experts)
    k.router(x, w, z, ids, weights, groups[0], groups[1], **how)
    want = x.double() @ w.double().T
    # an order of `width` 32-bit sums: each is off by a share of the products' absolute values
    bound = (x.double().abs() @ w.double().abs().T) * (2.0 ** -23) * max(4.0, width ** 0.5)
    assert ((z.double() - want).abs() <= bound).all()
    _, ids2, weights2 = made()
    k.router_topk(z, ids2, weights2, groups[0], groups[1], **how)
    assert torch.equal(ids, ids2) and torch.equal(weights, weights2)
    if rows > 1 and outputs * width <= k.ROUTER_FUSED_WEIGHT and width % 8 == 0 and experts <= 64:        # a token's logits are its own
        z1, ids1, weights1 = (t[:1] for t in made())
        k.router(x[1:2].clone(), w, z1, ids1, weights1, groups[0], groups[1], **how)
        assert torch.equal(z1, z[1:2]) and torch.equal(ids1, ids[1:2])


# (rows on either side of where four tokens share a workgroup, of a last workgroup that is not full, and of where the product used to
# go to the vendor library: 2^25 products)
@pytest.mark.parametrize("outputs,width,top", [(8, 2048, 2), (20, 2048, 4), (8, 4096, 2), (65, 520, 8), (16, 1000, 3), (5, 8, 2)])
def test_a_tokens_logits_and_choice_are_the_same_in_every_step(outputs, width, top):
    gen = torch.Generator().manual_seed(outputs + width)
    k = Kernels(torch.bfloat16, routed=True)
    x, w = torch.randn((2306, width), generator=gen).bfloat16().cuda(), (torch.randn((outputs, width), generator=gen) * 0.05).bfloat16().cuda()
    experts = min(outputs, 64)
    got = []
    for rows in (2306, 1, 3, 17, 767, 768, 769, 819, 820, 1024, 2047, 2048, 2049):
        z = torch.full((rows, outputs), float("nan"), device="cuda")
        ids, weights = torch.full((rows, top), -1, dtype=torch.int32, device="cuda"), torch.full((rows, top), float("nan"), device="cuda")
        k.router(x[:rows], w, z, ids, weights, renormalize=True, score="softmax", group_score="best", experts=experts)
        got.append((z, ids, weights))
        assert all(torch.equal(part, whole[:rows]) for part, whole in zip(got[-1], got[0])), rows


# What the rule for a model that routes asks of the router itself: its logits are no further from 64 bits than those of the product that
# the other models' projections take, and no more tokens choose other experts than the exact logits would.
@pytest.mark.parametrize("outputs,width,top", [(8, 2048, 2), (20, 2048, 4), (16, 1024, 4), (8, 4096, 2)])
@pytest.mark.parametrize("rows,seeds", [(16, 40), (48, 30), (820, 6), (2049, 4)])
def test_one_launch_is_as_exact_as_the_product_and_chooses_as_the_exact_logits_do(outputs, width, top, rows, seeds):
    k = Kernels(torch.bfloat16, routed=True)
    error, others = [0.0, 0.0], [0, 0]
    for seed in range(seeds):
        gen = torch.Generator(device="cuda").manual_seed(1000 * rows + seed)
        draw = lambda *shape: torch.randn(shape, generator=gen, device="cuda")  # noqa: E731
        x, w = draw(rows, width).bfloat16(), (0.05 * draw(outputs, width)).bfloat16()
        want = x.double() @ w.double().T
        chosen = want.topk(top, 1).indices.sort(1).values
        z, ids, weights = torch.empty(rows, outputs, device="cuda"), torch.empty(rows, top, dtype=torch.int32, device="cuda"), torch.empty(rows, top, device="cuda")
        for i in range(2):
            if i == 0:
                k.router(x, w, z, ids, weights, score="softmax", group_score="best")
            else:
                k.gemm(x, w, z)
                k.router_topk(z, ids, weights, score="softmax", group_score="best")
            error[i] += float(((z.double() - want) ** 2).sum())
            others[i] += int((ids.long().sort(1).values != chosen).any(1).sum())
    assert error[0] <= error[1] and others[0] <= others[1]
