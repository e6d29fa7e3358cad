"""The token log-probability kernels where rows are cut into parts and where they are not aligned."""
import pytest
import torch

from torchtitan_amd import ops

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("vocab", [1, 7, 8, 16384, 16385, 40011])
@pytest.mark.parametrize("splits", [1, 2, 5])
@pytest.mark.parametrize("offset", [0, 1, 6])
def test_log_probs_of_cut_and_unaligned_rows(device, vocab, splits, offset, monkeypatch):
    """Against float64 log-softmax: log-probabilities within 1e-5 (float32 sums of up to 40 011
    terms), the bf16 gradient within one step of bf16 (2^-7 of the value); parts without any
    element and a row of -inf logits but one included."""
    rows = 5
    g = torch.Generator(device=device).manual_seed(vocab + splits)
    buf = (torch.randn(rows * (vocab + 3) + offset, generator=g, device=device) * 4).to(torch.bfloat16)
    logits = buf[offset:].view(rows, vocab + 3)[:, :vocab]
    target = torch.randint(0, vocab, (rows,), generator=g, device=device)
    logits[1] = float("-inf")
    logits[1, target[1]] = 2.5
    monkeypatch.setattr(ops, "_logprob_splits", lambda r, v: splits)
    lp, lse = ops.token_logprob_fwd(logits, target)
    want = torch.log_softmax(logits.double(), dim=-1)
    assert (lp.double() - want.gather(1, target[:, None])[:, 0]).abs().max() <= 1e-5
    assert (lse.double() - torch.logsumexp(logits.double(), dim=-1)).abs().max() <= 1e-5
    grad = torch.randn(rows, generator=g, device=device)
    d = ops.token_logprob_bwd(logits, target, lse, grad).double()
    exact = -want.exp()
    exact[torch.arange(rows), target] += 1
    exact *= grad[:, None].double()
    assert ((d - exact).abs() <= exact.abs() * 2.0 ** -7 + 1e-6).all()


@pytest.mark.parametrize("splits", [1, 3])
@pytest.mark.parametrize("lo,hi", [(0, 8), (2400, 2408), (4096, 4104), (40000, 40008), (40008, 40011), (0, 40011)])
def test_nan_logits_are_not_lost(device, lo, hi, splits, monkeypatch):
    """A lane whose first piece is all NaN, in every place that reads one: the row is NaN, its neighbour
    is not, and -inf beside the NaN changes nothing."""
    logits = torch.randn((3, 40011), device=device).to(torch.bfloat16)
    logits[2] = float("-inf")
    logits[::2, lo:hi] = float("nan")
    target = torch.full((3,), 17, device=device)
    monkeypatch.setattr(ops, "_logprob_splits", lambda r, v: splits)
    lp, lse = ops.token_logprob_fwd(logits, target)
    assert lp.isnan().tolist() == [True, False, True] and lse.isnan().tolist() == [True, False, True]


@pytest.mark.parametrize("vocab", [8, 1001, 16384])
def test_log_probs_of_rows_that_overlap(device, vocab):
    """One row expanded to several, from any element, and a column seen as a row: as their contiguous copies."""
    base = torch.randn(vocab + 1, device=device).to(torch.bfloat16)
    for logits in (base[:vocab].expand(3, -1), base[1:].expand(3, -1), base[1:, None].t()):
        target = torch.arange(logits.shape[0], device=device) % vocab
        results = []
        for t in (logits, logits.contiguous().view(-1).clone().view(logits.shape)):
            lp, lse = ops.token_logprob_fwd(t, target)
            results.append((lp, lse, ops.token_logprob_bwd(t, target, lse, torch.ones_like(lp))))
        assert all(torch.equal(a, b) for a, b in zip(*results))


@pytest.mark.parametrize("vocab", [1, 7, 8, 1000, 2047, 8192, 8200, 12288, 12289])
@pytest.mark.parametrize("rows", [512, 513])
def test_log_probs_of_many_short_rows(device, rows, vocab):
    """On either side of the rows that half a workgroup takes: as above, within 1e-5."""
    g = torch.Generator(device=device).manual_seed(vocab)
    logits = (torch.randn((rows, vocab), generator=g, device=device) * 4).to(torch.bfloat16)
    logits[1], logits[3, 0] = float("-inf"), float("nan")
    logits[1, -1] = 0.5
    target = torch.randint(0, vocab, (rows,), generator=g, device=device)
    target[1] = vocab - 1
    lp, lse = ops.token_logprob_fwd(logits, target)
    want = torch.log_softmax(logits.double(), dim=-1).gather(1, target[:, None])[:, 0]
    fine = torch.arange(rows, device=device) != 3
    assert lp[3].isnan() and lse[3].isnan() and (lp.double() - want)[fine].abs().max() <= 1e-5
    assert (lse.double() - torch.logsumexp(logits.double(), dim=-1))[fine].abs().max() <= 1e-5


def test_parts_follow_the_number_of_rows():
    assert ops._logprob_splits(16, 151936) == 12 and ops._logprob_splits(64, 151936) == 4
    assert ops._logprob_splits(256, 151936) == 1 and ops._logprob_splits(16, 8192) == 1
