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
    if rows > 1 and rows * outputs * width <= k.ROUTER_FUSED_WORK and width % 8 == 0 and experts <= 64:        # a token's logits are its own
        z1, ids1, weights1 = (t[:1] for t in made())
        k.router(x[1:2].clone(), w, z1, ids1, weights1, groups[0], groups[1], **how)
        assert torch.equal(z1, z[1:2]) and torch.equal(ids1, ids[1:2])
