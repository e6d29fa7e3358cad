"""Products of a few rows against float64 products of the dequantized operands the casts write, and
converted modules on either side of the row limit."""
import pytest
import torch
import torch.nn as nn

from torchtitan_amd import _lib, ops
from torchtitan_amd.modules import FeedForward, Linear
from torchtitan_amd.protocols import ModelConvertersContainer
from torchtitan_amd.quantization.mx import MXFP8Converter

pytestmark = pytest.mark.gpu


def _values(rows, cols, device, seed):
    g = torch.Generator(device=device).manual_seed(seed)
    x = torch.randn((rows, cols), generator=g, device=device)
    x[torch.rand((rows, cols), generator=g, device=device) < 1e-2] *= 100
    return x.to(torch.bfloat16)


def _dequantized(x, mode):
    """float64 values of the row-wise cast of x."""
    return ops.mx_dequant(ops.to_mx_dim0(x, mode)).double()


def _check(got, xd, wd):
    """One rounding to bf16 (2^-8 of the value) and the sums: the matrix core aligns the products of a step to the
    largest before it adds them, which costs up to 1.2e-4 of the sum of magnitudes on such inputs, measured on the
    128 x 128 tile kernel over contractions of 32 to 14336; 2^-12 is twice that."""
    want = xd @ wd.t()
    assert ((got.double() - want).abs() <= want.abs() * 2.0 ** -8 + (xd.abs() @ wd.abs().t()) * 2.0 ** -12).all()


# rows around the kernel's 16-row tiles; contractions of one step to more than two rounds of the waves, with
# 32, 64 and 96 behind the last whole step; columns around its 16 and the scales' 128
@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("M", [1, 15, 16, 17, 32, 33, 48, 49, 64])
@pytest.mark.parametrize("K,N", [(32, 1), (128, 16), (224, 17), (1024, 130), (1120, 96), (2176, 272), (3136, 257),
                                 (256, 6160), (160, 12304)])
def test_few_rows_products(device, M, K, N, mode):
    x, w, w2 = _values(M, K, device, M), _values(N, K, device, N), _values(N, K, device, N + 1)
    wq, w2q = (ops.to_operands(t, mode, True, False, 128)[0] for t in (w, w2))
    xd, wd = _dequantized(x, mode), _dequantized(w, mode)
    xq = ops.to_operands(x, mode, True, False, 128)[0]
    one = ops.mx_gemm_nt(xq, wq)
    _check(one, xd, wd)
    if K <= 128:  # one step: nothing is added behind the matrix core
        _lib.load().mx_debug_force_kernel(2)
        try:
            assert torch.equal(ops.mx_gemm_nt(xq, wq), one)
        finally:
            _lib.load().mx_debug_force_kernel(0)
    if M > ops.FEW_ROWS:  # too many rows to be cast by every workgroup
        with pytest.raises(_lib.MXLibraryError):
            ops.mx_few_rows(x, wq, mode)
        return
    assert torch.equal(ops.mx_few_rows(x, wq, mode), one)  # the same steps in the same order
    both = ops.mx_few_rows(x, wq, mode, w2q)
    _check(both[0], xd, wd)
    _check(both[1], xd, _dequantized(w2, mode))


def test_few_rows_of_a_view_and_of_special_values(device):
    x, w = _values(30, 512, device, 1), _values(64, 256, device, 2)
    x[3, 70], x[5, 200], x[7, 33] = float("nan"), float("inf"), float("-inf")
    wq = ops.to_operands(w, "rceil", True, False)[0]
    for view in (x[:, 128:384], x[::2, 4:260], x[:, :256]):
        got = ops.mx_few_rows(view, wq, "rceil")
        want = ops.mx_gemm_nt(ops.to_operands(view.contiguous(), "rceil", True, False)[0], wq)
        assert torch.equal(got.nan_to_num(7.0, 8.0, 9.0), want.nan_to_num(7.0, 8.0, 9.0))
    with pytest.raises(ValueError):
        ops.mx_few_rows(x, wq, "rceil")


@pytest.mark.parametrize("tokens", [1, 32, 33, 64, 65])
def test_modules_without_gradients(device, tokens):
    """A forward without gradients equals the training forward up to float32 summation order."""
    for module, fqn in ((Linear.Config().build(in_features=192, out_features=160), "block"),
                        (FeedForward.Config(hidden_dim=384).build(dim=192), "block")):
        holder = nn.Module()
        holder.block = module
        ModelConvertersContainer.Config(converters=[MXFP8Converter.Config(fqns=[fqn])]).build(
            parallel_dims=None, model_compile_enabled=False).convert(holder)
        holder.to(device).to(torch.bfloat16)
        with torch.no_grad():
            for p in holder.parameters():
                p.copy_(_values(*p.shape, device, 3) * 0.05)
        x = _values(tokens, 192, device, tokens)[None]
        want = holder.block(x.requires_grad_(True)).detach()
        with torch.no_grad():
            got = holder.block(x.detach())
        assert got.shape == want.shape
        # a last bit of a hidden value may move one e4m3 code of 1/16 at most behind it
        assert (got - want).float().norm() <= 2e-2 * want.float().norm()


def test_cached_casts_of_another_form(device):
    """A dense cached weight cast, as a traced forward leaves it, serves an eager forward without gradients."""
    from torchtitan_amd import mx_tensor

    cfg = mx_tensor.MXFP8Config(cache_weight_casts=True)
    x, w = _values(5, 256, device, 1), _values(128, 256, device, 2)
    mx_tensor._weight_cache.clear()
    want, _, _ = mx_tensor._linear_forward(x, w, cfg, False, False)
    mx_tensor._weight_cache.clear()
    dense, _ = mx_tensor._cast_weight(w, cfg.scale_mode, True, cfg, whole_blocks=False)
    assert type(dense) is not ops.Operand
    got, _, _ = mx_tensor._linear_forward(x, w, cfg, False, False)
    mx_tensor._weight_cache.clear()
    assert torch.equal(got, want)


@pytest.mark.parametrize("K", [256, 512])
@pytest.mark.parametrize("N", [16384, 16400])
def test_products_on_either_side_of_the_widest(device, N, K):
    """Where few rows go to workgroups of their own or to tiles."""
    w = _values(N, K, device, 1) * 0.1
    wq, wd = ops.to_operands(w, "rceil", True, False, 128)[0], _dequantized(w, "rceil")
    for M in (1, 16, 17, 64):
        x = _values(M, K, device, M)
        _check(ops.mx_gemm_nt(ops.to_operands(x, "rceil", True, False, 128)[0], wq), _dequantized(x, "rceil"), wd)
        with torch.no_grad():
            assert ops.few_rows_ok(x, N) == (M <= ops.FEW_ROWS and N <= 16384)
