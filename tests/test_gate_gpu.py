"""The gate kernels against float64: tile edges of tokens (16 and 32 per workgroup, 32 per step of the weight
gradient), experts (16, 32, 64 and 128 per variant) and columns (128 per wave)."""
import pytest
import torch

from torchtitan_amd import ops
from torchtitan_amd.modules.moe import MoE
from torchtitan_amd.mx_blocks import gate_fusable, mx_gate

pytestmark = pytest.mark.gpu


def _within_bf16(got, want, noise):
    """Half a step of bf16 (eight significant bits: at most 2^-8 of the value) and the float32 sum's own
    error."""
    return bool(((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + noise).all())


@pytest.mark.parametrize("tokens,experts,dim", [(1, 8, 128), (15, 16, 256), (17, 24, 384), (33, 32, 640), (130, 40, 128),
                                                (97, 64, 1024), (300, 72, 2048), (129, 128, 512), (4100, 8, 128),
                                                (4129, 128, 256), (5003, 56, 1152), (9000, 128, 2048)])
def test_gate_against_float64(device, tokens, experts, dim):
    """Sums of n float32 products: error below 2^-24 sqrt(n) times the root of the summed squares, with a
    factor of 8 for the largest of up to 10^7 entries."""
    g = torch.Generator(device=device).manual_seed(tokens + experts + dim)
    x = torch.randn((tokens, dim), generator=g, device=device).bfloat16().requires_grad_(True)
    w = (torch.randn((experts, dim), generator=g, device=device) * 0.02).bfloat16().requires_grad_(True)
    dl = torch.randn((tokens, experts), generator=g, device=device) * 1e-3
    base = torch.randn((tokens, dim), generator=g, device=device).bfloat16() * 1e-4
    logits, x2 = mx_gate(x, w)
    assert torch.equal(x2, x) and logits.dtype == torch.float32
    want = x.detach().double() @ w.detach().double().T
    eps = 8 * 2.0 ** -24
    assert (logits.double() - want).abs().max() <= eps * dim ** 0.5 * 0.02 * dim ** 0.5
    dx, dw = torch.autograd.grad((logits, x2), (x, w), (dl, base))
    plain = dl.double() @ w.detach().double()
    alone = ops.gate_dx(dl, w.detach())
    assert torch.equal(dx, alone + base)
    assert _within_bf16(dw, dl.double().T @ x.detach().double(), eps * tokens ** 0.5 * 1e-3 * tokens ** 0.5)
    assert _within_bf16(alone, plain, eps * experts ** 0.5 * 2e-5 * experts ** 0.5)
    # without a gradient into the activation, and without one from behind
    (only,) = torch.autograd.grad(mx_gate(x.detach(), w)[0], w, dl)
    assert torch.equal(only, dw)
    (behind,) = torch.autograd.grad(mx_gate(x, w)[1], x, base)
    assert torch.equal(behind, base)


@pytest.mark.parametrize("experts,dim", [(8, 2048), (32, 4096), (64, 2048), (72, 2048), (16, 1024), (128, 384)])
@pytest.mark.parametrize("tokens", [300, 4100, 9001])
def test_logits_do_not_depend_on_where_a_token_stands(device, tokens, experts, dim):
    """Bit for bit the same anywhere in a batch and in a batch of another size, in every order of the
    contraction that workgroups take."""
    g = torch.Generator(device=device).manual_seed(experts + dim)
    some = torch.randn((50, dim), generator=g, device=device).bfloat16()
    w = (torch.randn((experts, dim), generator=g, device=device) * 0.02).bfloat16()
    which = torch.randint(0, 50, (tokens,), generator=g, device=device)
    assert torch.equal(ops.gate_logits(some[which], w), ops.gate_logits(some, w)[which])


def test_gate_keeps_infinite_gradients(device):
    dl = torch.zeros((16, 8), device=device)
    dl[3, 2], dl[5, 1] = float("inf"), float("nan")
    w = torch.ones((8, 128), dtype=torch.bfloat16, device=device)
    dx = ops.gate_dx(dl, w)
    assert bool(torch.isposinf(dx[3]).all()) and bool(torch.isnan(dx[5]).all())
    assert not dx[:3].any() and not dx[4].any() and not dx[6:].any()


def test_gate_gradient_onto_an_expanded_row(device):
    dl, w = torch.randn((40, 8), device=device), torch.randn((8, 128), device=device).bfloat16()
    base = torch.randn((1, 128), device=device).bfloat16().expand(40, -1)
    assert torch.equal(ops.gate_dx(dl, w, base), ops.gate_dx(dl, w, base.contiguous()))


@pytest.mark.parametrize("change", ["bias", "hook", "float32 weight", "experts", "dim"])
def test_gate_leaves_other_gates_alone(device, change):
    """Calls that the kernels do not take, or that somebody listens to, go through the gate module."""
    experts, dim = (12, 256) if change == "experts" else (8, 96) if change == "dim" else (8, 256)
    cfg = MoE.Config(num_experts=experts, num_shared_experts=0, hidden_dim=64, top_k=2, gate_bias=change == "bias")
    with torch.device(device):
        moe = MoE(cfg, dim=dim)
    gate = moe.router.gate.to(torch.float32 if change == "float32 weight" else torch.bfloat16)
    x = torch.randn((20, dim), device=device).bfloat16()
    if change != "hook":
        assert not gate_fusable(x, gate.weight, gate.bias)
        return
    from torchtitan_amd.modules.linear import Linear
    from torchtitan_amd.modules.moe import _stock

    assert gate_fusable(x, gate.weight, gate.bias) and _stock(gate, Linear)
    gate.register_forward_hook(lambda *a: None)
    assert not _stock(gate, Linear)
