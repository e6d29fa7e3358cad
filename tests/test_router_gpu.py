"""The routing kernels: scores, top-k choice, weights and their gradient against torch in float64, the
placement of the pairs against the plan from a stable sort."""
import pytest
import torch

from torchtitan_amd import ops
from torchtitan_amd.mx_blocks import mx_route_topk

pytestmark = pytest.mark.gpu


def _reference(logits, bias, k, softmax, norm, scale):
    x = logits.double()
    s = torch.softmax(x, dim=1) if softmax else torch.sigmoid(x)
    choice = s if bias is None else s + bias.double()
    selected = torch.topk(choice, k, dim=1).indices
    w = s.gather(1, selected)
    if norm:
        w = w / (w.sum(dim=1, keepdim=True) + 1e-20)
    return selected, w * scale, choice


# tokens around a workgroup's 16 and a wave's share of it; experts around 64 per register; every k limit
@pytest.mark.parametrize("tokens,experts,k", [(1, 2, 1), (15, 8, 2), (16, 64, 8), (17, 65, 6), (300, 128, 8),
                                              (33, 129, 16), (70, 512, 16), (5, 16, 16)])
@pytest.mark.parametrize("softmax,norm,with_bias", [(True, True, False), (True, False, True), (False, True, True),
                                                    (False, False, False)])
def test_routing_against_float64(device, tokens, experts, k, softmax, norm, with_bias):
    """Weights within 2e-6 (float32 scores and sums of up to 512 terms), the same choice wherever the
    float64 scores are further than 1e-6 apart, the gradient within 1e-5 of its row's norm."""
    g = torch.Generator(device=device).manual_seed(tokens + experts + k)
    logits = (torch.randn((tokens, experts), generator=g, device=device) * 2).requires_grad_(True)
    bias = torch.randn(experts, generator=g, device=device) * 0.1 if with_bias else None
    top, selected, counts, _ = mx_route_topk(logits, bias, k, softmax, norm, 1.5)
    want_sel, want_top, choice = _reference(logits, bias, k, softmax, norm, 1.5)
    picked = choice.gather(1, selected)
    assert (picked - choice.gather(1, want_sel)).abs().max() <= 1e-6
    assert bool((picked[:, :-1] >= picked[:, 1:] - 1e-6).all())
    assert all(len(set(row)) == k for row in selected.tolist())
    s = torch.softmax(logits.double(), 1) if softmax else torch.sigmoid(logits.double())
    w = s.gather(1, selected)
    w = (w / (w.sum(1, keepdim=True) + 1e-20) if norm else w) * 1.5
    assert (top.double() - w).abs().max() <= 2e-6
    assert torch.equal(counts, torch.bincount(selected.flatten(), minlength=experts))
    dtop = torch.randn((tokens, k), generator=g, device=device)
    (got,) = torch.autograd.grad(top, logits, dtop)
    (want,) = torch.autograd.grad(w, logits, dtop.double())
    assert (got.double() - want).norm() <= 1e-5 * want.norm() + 1e-7


@pytest.mark.parametrize("k", [1, 2, 3, 5, 8, 11, 16])
@pytest.mark.parametrize("softmax", [True, False])
def test_weights_are_normalised_by_a_tree_sum(device, k, softmax):
    """Bit for bit the scores over their sum, pairs of neighbours added first: its error grows with the
    logarithm of k, that of a running sum with k."""
    logits = torch.randn((3000, 128), generator=torch.Generator(device=device).manual_seed(k), device=device) * 2
    scores = ops.route_topk(logits, None, k, softmax, False, 1.0)[0]
    total = torch.nn.functional.pad(scores, (0, 16 - k))
    while total.shape[1] > 1:
        total = total[:, 0::2] + total[:, 1::2]
    assert torch.equal(ops.route_topk(logits, None, k, softmax, True, 1.0)[0], scores / (total + 1e-20))


def test_equal_scores_go_to_the_lower_experts(device):
    top, selected, counts, _ = ops.route_topk(torch.zeros((3, 130), device=device), None, 4, True, False, 1.0)
    assert selected.tolist() == [[0, 1, 2, 3]] * 3 and counts.tolist() == [3] * 4 + [0] * 126
    assert torch.allclose(top, torch.full((3, 4), 1 / 130, device=device))


@pytest.mark.parametrize("sign", [0x7FC00000, 0x7FC00000 - 2 ** 31])
def test_nan_is_above_every_score(device, sign):
    """Of either sign, as torch.topk orders it; the rest in falling order behind it."""
    bias = torch.zeros(70, device=device)
    bias.view(torch.int32)[66] = sign
    logits = torch.arange(70, dtype=torch.float32, device=device).mul(0.1).expand(3, 70).contiguous()
    _, selected, counts, _ = ops.route_topk(logits, bias, 3, False, False, 1.0)
    assert selected.tolist() == [[66, 69, 68]] * 3 and counts.sum().item() == 9
    assert torch.topk(torch.sigmoid(logits) + bias, 3, dim=1).indices.tolist() == selected.tolist()


@pytest.mark.parametrize("tokens,experts,k", [(1, 2, 1), (17, 8, 2), (300, 65, 4), (1000, 128, 8), (40, 300, 16)])
@pytest.mark.parametrize("alignment,multiple", [(32, 1), (32, 128), (8, 8)])
def test_plan_equals_the_plan_from_a_stable_sort(device, tokens, experts, k, alignment, multiple):
    g = torch.Generator(device=device).manual_seed(7 * tokens + experts)
    # a skewed choice: some experts get most tokens, some none
    logits = torch.randn((tokens, experts), generator=g, device=device)
    logits += 2 * torch.randn((1, experts), generator=g, device=device)
    top, selected, counts, block_counts = ops.route_topk(logits, None, k, False, False, 1.0)
    got = ops.route_fill(selected, top, counts, block_counts, alignment, multiple)
    order = torch.argsort(selected.flatten(), stable=True)
    want = ops.moe_route_plan(counts, order, top.flatten(), k, alignment, multiple)
    for a, b in zip(got, want):
        assert torch.equal(a.flatten(), b)


@pytest.mark.parametrize("softmax,norm", [(True, True), (True, False), (False, True), (False, False)])
def test_routing_twice_differentiated_and_transformed(device, softmax, norm):
    """The gradient of the weights can be differentiated, and transforms take the tensor operations."""
    from torchtitan_amd import mx_blocks

    g = torch.Generator(device=device).manual_seed(5)
    logits = torch.randn((7, 16), generator=g, device=device, requires_grad=True)
    v, u = (torch.randn((7, n), generator=g, device=device) for n in (4, 16))
    top, selected, *_ = mx_blocks.mx_route_topk(logits, None, 4, softmax, norm, 1.5)
    plain = mx_blocks._route_weights(logits, selected, softmax, norm, 1.5)
    second = []
    for t in (top, plain):
        (first,) = torch.autograd.grad(t, logits, v, create_graph=True)
        second.append(torch.autograd.grad(first, logits, u)[0])
    torch.testing.assert_close(second[0], second[1], rtol=1e-5, atol=1e-6)
    assert mx_blocks.route_fusable(logits, 4)
    seen = []
    torch.func.vmap(lambda t: (seen.append(mx_blocks.route_fusable(t, 4)), t)[1])(logits.detach()[None])
    with torch.autograd.forward_ad.dual_level():
        seen.append(mx_blocks.route_fusable(logits, 4))
    assert seen == [False, False]


def test_forward_without_gradients_refuses_tangents(device):
    """A converted linear has no forward-mode derivative: with gradients off it says so, too."""
    from torchtitan_amd import mx_tensor

    x = torch.randn((4, 64), device=device, dtype=torch.bfloat16)
    w = torch.randn((32, 64), device=device, dtype=torch.bfloat16)
    with torch.no_grad(), torch.autograd.forward_ad.dual_level():
        dual = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        with pytest.raises(Exception):
            mx_tensor.mx_linear(dual, w, None, mx_tensor.MXFP8Config())


@pytest.mark.parametrize("bias", ["row", "one value", "per token", "one per token", "host value", "bf16"])
def test_a_bias_that_broadcasts(device, bias):
    """Whatever can be added to the scores steers the choice as the sum does."""
    from torchtitan_amd.modules.moe import MoE

    g = torch.Generator(device=device).manual_seed(2)
    with torch.device(device):
        router = MoE(MoE.Config(num_experts=16, num_shared_experts=0, hidden_dim=64, top_k=3, score_func="sigmoid"),
                     dim=128).router
    x = torch.randn((20, 128), generator=g, device=device)
    rn = lambda *shape: torch.randn(shape, generator=g, device=device) * 0.3
    b = {"row": rn(1, 16), "one value": rn(), "per token": rn(20, 16), "one per token": rn(20, 1),
         "host value": torch.tensor(0.5), "bf16": rn(16).bfloat16()}[bias]
    top, selected, counts = router(x, b)
    scores = torch.sigmoid(x @ router.gate.weight.t())
    want = torch.topk(scores + b, 3, dim=1).indices
    assert torch.equal(selected.sort(dim=1).values, want.sort(dim=1).values)
    assert counts.sum().item() == 60 and top.shape == (20, 3)
