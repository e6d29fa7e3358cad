"""Casts and dequantization of lists of tensors against the single-tensor kernels."""
import pytest
import torch

from torchtitan_amd import ops

pytestmark = pytest.mark.gpu


def _tensors(device, dtype, n):
    g = torch.Generator(device=device).manual_seed(n)
    # one block, around a workgroup's 8192 elements, a stack, and no element at all
    shapes = [(1, 32), (3, 64), (64, 128), (257, 32), (2, 40, 96), (0, 64), (130, 1056)]
    out = []
    for i in range(n):
        t = torch.randn(shapes[i % len(shapes)], generator=g, device=device) * 10.0 ** (i % 5 - 2)
        if t.numel() > 64:
            t.view(-1)[::77] = float("nan") if i % 3 == 0 else float("-inf")
        out.append(t.to(dtype))
    return out


@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("n", [1, 7, 48, 49, 100])  # around the 48 entries of a launch's table
def test_list_casts_equal_single_casts(device, mode, dtype, n):
    tensors = _tensors(device, dtype, n)
    many = ops.to_mx_rows_many(tensors, mode)
    back = ops.mx_dequant_many(many)
    for t, q, b in zip(tensors, many, back):
        assert q.codes.shape == t.shape and q.scales.shape == (*t.shape[:-1], t.shape[-1] // 32) and b.shape == t.shape
        if t.numel() == 0:
            continue
        one = ops.to_mx_dim0(t.to(torch.bfloat16).reshape(-1, t.shape[-1]), mode)
        assert torch.equal(q.codes.view(one.codes.shape), one.codes)
        assert torch.equal(q.scales.view(one.scales.shape), one.scales)
        assert torch.equal(b.view(one.codes.shape).view(torch.int16), ops.mx_dequant(one).view(torch.int16))


def test_lists_reject_what_they_cannot_take(device):
    assert ops.to_mx_rows_many([]) == [] and ops.mx_dequant_many([]) == []
    with pytest.raises(ValueError):
        ops.to_mx_rows_many([torch.zeros((2, 48), device=device, dtype=torch.bfloat16)])
    with pytest.raises(TypeError):
        ops.to_mx_rows_many([torch.zeros((2, 64), device=device, dtype=torch.float16)])
    q = ops.to_mx_dim0(torch.zeros((2, 64), device=device, dtype=torch.bfloat16), "floor", ops.MX_SCALES_MFMA)
    with pytest.raises(ValueError):
        ops.mx_dequant_many([q])
