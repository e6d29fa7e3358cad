"""Operands and converted modules over token counts and sizes that are no multiple of the format's
32-element blocks or of the GEMM's 128-deep ones: the casts write zeros up to whole blocks, which
changes no product, so everything equals the same call on a tensor with zero rows appended."""
import pytest
import torch
import torch.nn as nn

from torchtitan_amd import mx_tensor, ops
from torchtitan_amd.mx_blocks import feed_forward_fusable
from torchtitan_amd.modules import FeedForward, Linear
from torchtitan_amd.protocols import ModelConvertersContainer
from torchtitan_amd.quantization.mx import MXFP8Converter

pytestmark = pytest.mark.gpu

L = ops.MX_SCALES_MFMA
# one row, around a block of 32, around a tile of 128, several tiles with remainders
SIZES = [(1, 32), (31, 96), (32, 128), (33, 64), (127, 160), (128, 256), (129, 96), (300, 264), (259, 1184)]


def _values(rows, cols, device, seed=0):
    g = torch.Generator(device=device).manual_seed(seed)
    x = torch.randn((rows, cols), generator=g, device=device)
    x[torch.rand((rows, cols), generator=g, device=device) < 1e-2] *= 100
    return x.to(torch.bfloat16)


def _zero_padded(x, rows, cols):
    out = torch.zeros((rows, cols), dtype=x.dtype, device=x.device)
    out[:x.shape[0], :x.shape[1]] = x
    return out


def _check(q, rows, padded, mode):
    """`q`: an operand of `rows` rows; `padded`: the bf16 matrix it must hold, contraction in whole blocks."""
    want = ops.to_mx_dim0(padded, mode)
    assert torch.equal(q.codes, want.codes[:rows])
    assert torch.equal(ops.scale_unlayout(q.scales, rows, padded.shape[1] // 32), want.scales[:rows])


def _up(n, m=128):
    return -(-n // m) * m


@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("rows,cols", SIZES)
@pytest.mark.parametrize("pad", [0, 128])
def test_operands_hold_the_matrix_and_zeros(device, rows, cols, mode, pad):
    x = _values(rows, cols, device, rows + cols)
    by_row, by_col = ops.to_operands(x, mode, pitch_pad=pad)
    assert by_row.codes.shape == (rows, _up(cols)) and by_col.codes.shape == (cols, _up(rows))
    _check(by_row, rows, _zero_padded(x, rows, _up(cols)), mode)
    _check(by_col, cols, _zero_padded(x.t(), cols, _up(rows)).contiguous(), mode)
    only_row, none = ops.to_operands(x, mode, cols=False, pitch_pad=pad)
    assert none is None and torch.equal(only_row.codes, by_row.codes) and torch.equal(only_row.scales, by_row.scales)
    none, only_col = ops.to_operands(x, mode, rows=False, pitch_pad=pad)
    assert none is None and torch.equal(only_col.codes, by_col.codes) and torch.equal(only_col.scales, by_col.scales)
    # rows that are not 16-byte aligned are copied first
    shifted = torch.zeros(rows * cols + 4, dtype=x.dtype, device=device)[4:].view(rows, cols).copy_(x)
    assert torch.equal(ops.to_operands(shifted, mode)[0].codes, by_row.codes)


@pytest.mark.parametrize("rows,cols", SIZES)
def test_float32_input_is_rounded_like_a_conversion(device, rows, cols):
    x = _values(rows, cols, device, 3).float()
    x += x.abs() * 2.0 ** -9 * torch.rand_like(x)  # off the bf16 grid, ties and NaN among them
    x.view(-1)[::7] = x.view(-1)[::7].to(torch.bfloat16).float() * (1 + 2.0 ** -8)
    if rows * cols > 200:
        x.view(-1)[::97] = float("nan")
    for want, got in zip(ops.to_operands(x.to(torch.bfloat16), "rceil"), ops.to_operands(x, "rceil")):
        assert torch.equal(got.codes, want.codes) and torch.equal(got.scales, want.scales)
    shifted = torch.zeros(rows * cols + 1, device=device)[1:].view(rows, cols).copy_(x)
    assert torch.equal(ops.to_operands(shifted, "rceil")[1].codes, want.codes)


@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("rows,cols", SIZES)
def test_gate_and_norm_operands_equal_the_casts_of_their_values(device, rows, cols, mode):
    a, b, dg = (_values(rows, cols, device, s) for s in (1, 2, 3))
    ap, bp, dgp = (_zero_padded(t, _up(rows), _up(cols)) for t in (a, b, dg))
    _, _, g = ops.swiglu_to_mx_dim0_dim1(ap, bp, mode, L, want_g=True)
    by_row, by_col = ops.swiglu_to_operands(a, b, mode, pitch_pad=128)
    _check(by_row, rows, g[:rows], mode)
    _check(by_col, cols, g.t()[:cols].contiguous(), mode)
    only, none = ops.swiglu_to_operands(a, b, mode, cols=False)
    assert none is None and torch.equal(only.codes, by_row.codes) and torch.equal(only.scales, by_row.scales)
    _, _, grads = ops.swiglu_bwd_to_mx_dim0_dim1(dgp, ap, bp, mode, L, want_grads=True)
    for (r, c), t in zip(ops.swiglu_bwd_to_operands(dg, a, b, mode, pitch_pad=128), grads):
        _check(r, rows, t[:rows], mode)
        _check(c, cols, t.t()[:cols].contiguous(), mode)
    if cols % 32 == 0:
        w = _values(1, cols, device, 4)[0]
        _, _, rstd, y = ops.rms_norm_to_mx(_zero_padded(a, _up(rows, 32), cols), w, 1e-5, mode, L, want_y=True)
        r, c, rstd_r = ops.rms_norm_to_operands(a, w, 1e-5, mode)
        assert torch.equal(rstd_r, rstd[:rows])
        _check(r, rows, _zero_padded(y[:rows], rows, _up(cols)), mode)
        _check(c, cols, _zero_padded(y[:rows].t(), cols, _up(rows)).contiguous(), mode)


def _converted(module, device, **options):
    holder = nn.Module()
    holder.block = module
    ModelConvertersContainer.Config(converters=[MXFP8Converter.Config(fqns=["block"], **options)]).build(
        parallel_dims=None, model_compile_enabled=False).convert(holder)
    holder.to(device).to(torch.bfloat16)
    g = torch.Generator(device=device).manual_seed(5)
    with torch.no_grad():
        for p in holder.parameters():
            p.normal_(0.0, 0.05, generator=g)
    return module


def _step(module, x, dy):
    mx_tensor.clear_cast_cache()
    xi = x.clone().requires_grad_(True)
    y = module(xi)
    grads = torch.autograd.grad(y, [xi, *module.parameters()], dy)
    return [y.detach(), *grads]


@pytest.mark.parametrize("cache", [False, True])
@pytest.mark.parametrize("tokens,inner,outer", [(1, 128, 256), (45, 96, 160), (300, 256, 384), (517, 416, 272)])
def test_linear_over_any_number_of_tokens(device, tokens, inner, outer, cache):
    """Against the same linear with zero tokens appended up to a multiple of 128 (identical tiles and
    order of summation): every result bit for bit."""
    lin = _converted(Linear.Config().build(in_features=inner, out_features=outer), device, cache_weight_casts=cache)
    x, dy = _values(tokens, inner, device, 6), _values(tokens, outer, device, 7)
    whole = _up(tokens)
    want = _step(lin, _zero_padded(x, whole, inner), _zero_padded(dy, whole, outer))
    y, dx, dw = _step(lin, x, dy)
    assert torch.equal(y, want[0][:tokens]) and torch.equal(dx, want[1][:tokens]) and torch.equal(dw, want[2])
    with torch.no_grad():
        assert torch.equal(lin(x), y)


@pytest.mark.parametrize("tokens,dim,hidden", [(45, 96, 160), (300, 256, 512), (517, 160, 416)])
def test_feed_forward_over_any_number_of_tokens(device, tokens, dim, hidden):
    ff = _converted(FeedForward.Config(hidden_dim=hidden).build(dim=dim), device)
    x, dy = _values(tokens, dim, device, 8), _values(tokens, dim, device, 9)
    assert feed_forward_fusable(x, ff.w1.weight, ff.w2.weight, ff.w3.weight)
    whole = _up(tokens)
    want = _step(ff, _zero_padded(x, whole, dim), _zero_padded(dy, whole, dim))
    got = _step(ff, x, dy)
    for i, (g, w) in enumerate(zip(got, want)):
        assert torch.equal(g, w[:tokens] if i < 2 else w), i


@pytest.mark.parametrize("tokens", [1, 45, 256])
@pytest.mark.parametrize("block", ["linear", "ffn"])
def test_gradients_whose_rows_are_one_expanded_row(device, tokens, block):
    """The gradient behind a sum over tokens has stride 0 between its rows: the same as written out."""
    module = Linear.Config().build(in_features=128, out_features=160) if block == "linear" else \
        FeedForward.Config(hidden_dim=256).build(dim=128)
    module = _converted(module, device)
    x, row = _values(tokens, 128, device, 11), _values(1, 160 if block == "linear" else 128, device, 12)
    dy = row.expand(tokens, -1) if tokens > 1 else row.as_strided(row.shape, (0, 1))
    for got, want in zip(_step(module, x, dy), _step(module, x, dy.clone(memory_format=torch.contiguous_format))):
        assert torch.equal(got, want)


# tile counts around the walk's bands of 32 tile rows and strips of 2 (both forms) and of 2 and 32 (rows alone)
@pytest.mark.parametrize("tile_rows,tile_cols", [(32, 2), (33, 1), (33, 3), (31, 33), (3, 65), (65, 5),
                                                 (64, 4), (4, 64)])
def test_every_tile_of_the_walk_is_cast_once(device, tile_rows, tile_cols):
    rows, cols = 128 * tile_rows - 5, 128 * tile_cols - 32
    x = _values(rows, cols, device, tile_rows)
    by_row, by_col = ops.to_operands(x, "rceil")
    _check(by_row, rows, _zero_padded(x, rows, _up(cols)), "rceil")
    _check(by_col, cols, _zero_padded(x.t(), cols, _up(rows)).contiguous(), "rceil")
    only_row, _ = ops.to_operands(x, "rceil", cols=False)
    assert torch.equal(only_row.codes, by_row.codes) and torch.equal(only_row.scales, by_row.scales)


@pytest.mark.parametrize("mode", ["rceil", "floor"])
@pytest.mark.parametrize("pad", [0, 128])
def test_casts_of_a_list_equal_the_single_casts(device, mode, pad):
    """Matrices of uneven sizes and both types, a stack and an unaligned view in one launch of eight."""
    tensors = [_values(r, c, device, r) for r, c in [(1, 32), (129, 96), (4225, 128), (300, 264)]]
    tensors += [_values(257, 160, device, 5).float(), _values(64, 72, device, 6)[:, 4:68]]
    stacks = [_values(3 * 256, 128, device, 7).view(3, 256, 128), _values(2 * 128, 384, device, 8).view(2, 128, 384)]
    casts = ops.CastList(mode)
    got = [casts.add(t, pad) for t in tensors] + [casts.add_stack(t) for t in stacks]
    assert len(got) == ops.CAST_LIST
    with pytest.raises(ops._lib.MXLibraryError):
        casts.add(tensors[0])
    casts.launch()
    for t, pair in zip(tensors, got):
        for q, want in zip(pair, ops.to_operands(t, mode, pitch_pad=pad)):
            assert torch.equal(q.codes, want.codes) and torch.equal(q.scales, want.scales)
    for t, pair in zip(stacks, got[len(tensors):]):
        for q, want in zip(pair, ops.to_mx_dim0_dim1_batched(t, mode)):
            assert torch.equal(q.codes, want.codes) and torch.equal(q.scales, want.scales)
    with pytest.raises(ValueError):
        casts.add_stack(stacks[0][:, :32])
    q, _ = casts.add_stack(stacks[0].float())
    casts.launch()
    assert torch.equal(q.codes, got[len(tensors)][0].codes)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_activations_in_any_order(device, dtype):
    """Transposed and expanded inputs, as their contiguous copies: casts, lists of casts, and a converted linear
    under autocast, forward and backward."""
    from torchtitan_amd import mx_tensor

    g = torch.Generator(device=device).manual_seed(3)
    base = torch.randn((192, 96), generator=g, device=device).to(dtype)
    for x in (base.t(), base[:, :1].expand(192, 64), base[None].transpose(1, 2)[0], base.t()[::2, 64:], base[:, :1]):
        want = ops.to_operands(x.contiguous().clone(), "rceil")
        casts = ops.CastList("rceil")
        listed = casts.add(x)
        casts.launch()
        for q, p, w in zip(ops.to_operands(x, "rceil"), listed, want):
            assert torch.equal(q.codes, w.codes) and torch.equal(p.codes, w.codes)
    w = (torch.randn((64, 192), generator=g, device=device) * 0.05).to(dtype).requires_grad_(True)
    for x in (base.t(), base[None].transpose(1, 2)):
        out = []
        for t in (x, x.contiguous()):
            t = t.detach().requires_grad_(True)
            with torch.autocast("cuda", dtype=torch.bfloat16):
                y = mx_tensor.mx_linear(t, w, None, mx_tensor.MXFP8Config())
            out.append([y, *torch.autograd.grad(y, (t, w), torch.ones_like(y))])
            with torch.no_grad():
                out[-1].append(mx_tensor.mx_linear(t, w, None, mx_tensor.MXFP8Config()))
        for a, b in zip(*out):
            assert torch.equal(a, b)
