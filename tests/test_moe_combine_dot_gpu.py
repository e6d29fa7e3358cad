"""The combine that also takes the rows' dot products: the bits of the two separate kernels, at the edges
of its choices per wave and of a wave's 512 columns."""
import numpy as np
import pytest
import torch

from oracle import mx_oracle as mo
from torchtitan_amd import ops

from tests.helpers import bf16_from_bits, bits_of, randn_bits

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("tokens,k,cols", [(1, 1, 8), (5, 2, 512), (3, 3, 520), (67, 4, 1024), (33, 6, 264), (130, 8, 2048),
                                           (9, 9, 64), (21, 16, 768)])
def test_combine_dot_equals_combine_and_row_dot(device, tokens, k, cols):
    """Sum bit-exact against the oracle, dot products those of the row-dot kernel to the bit and within
    1e-5 of float64 (float32 sums of up to 2048 products); positions outside y count as nothing."""
    rng = np.random.default_rng(tokens + k)
    rows = tokens * k + 5
    y_bits, x_bits = randn_bits(rng, (rows, cols)), randn_bits(rng, (tokens, cols))
    pos = rng.permutation(rows)[: tokens * k].astype(np.int64).reshape(tokens, k)
    pos[0, 0], pos[-1, -1] = rows + 3, -1
    w = rng.random((tokens, k)).astype(np.float32)
    y, x = bf16_from_bits(y_bits, device), bf16_from_bits(x_bits, device)
    tp, tw = torch.from_numpy(pos).to(device), torch.from_numpy(w).to(device)
    token = torch.arange(tokens * k, device=device) // k
    dots = ops.moe_row_dot(y, tp.view(-1), x, token).view(tokens, k)
    ref = mo.moe_row_dot(y_bits, pos.reshape(-1), x_bits, token.cpu().numpy()).reshape(tokens, k)
    assert np.allclose(dots.cpu().numpy(), ref, rtol=1e-5, atol=1e-5 * np.sqrt(cols))
    for weights, want in ((tw, mo.moe_combine(y_bits, pos, w)), (None, mo.moe_combine(y_bits, pos, None))):
        out, got = ops.moe_combine_dot(y, tp, x, weights)
        assert np.array_equal(bits_of(out), want) and torch.equal(got, dots)
        assert np.array_equal(bits_of(ops.moe_combine(y, tp, weights)), want)
    out, got = ops.moe_combine_dot(y, tp, x, combine=False)
    assert out is None and torch.equal(got, dots)


@pytest.mark.parametrize("k", [0, 1, 2, 3, 4, 5, 6, 7, 8, 9, 11, 13, 16, 17, 26])
def test_combine_over_any_number_of_choices(device, k):
    """Bit-exact against the oracle in every number of rows that are asked for together, of one matrix and of two."""
    tokens, cols = 37, 264
    rng = np.random.default_rng(k)
    rows = tokens * k + 3
    y, y2 = (bf16_from_bits(randn_bits(rng, (rows, cols)), device) for _ in range(2))
    pos = rng.permutation(rows)[: tokens * k].astype(np.int64).reshape(tokens, k)
    if k:
        pos[0, 0], pos[-1, -1] = rows, -1
    w = rng.random((tokens, k)).astype(np.float32)
    tp, tw = torch.from_numpy(pos).to(device), torch.from_numpy(w).to(device)
    for weights, tweights in ((w, tw), (None, None)):
        assert np.array_equal(bits_of(ops.moe_combine(y, tp, tweights)), mo.moe_combine(bits_of(y), pos, weights))
        assert np.array_equal(bits_of(ops.moe_combine(y, tp, tweights, y2)), mo.moe_combine(bits_of(y + y2), pos, weights))


def test_no_rows_give_zeros(device):
    x = torch.ones((2, 64), dtype=torch.bfloat16, device=device)
    pos = torch.zeros((2, 3), dtype=torch.int64, device=device)
    spare = torch.empty((1, 64), dtype=torch.bfloat16, device=device)[:0]  # no rows, but an address
    out, dots = ops.moe_combine_dot(spare, pos, x)
    assert not out.any() and not dots.any()
