"""The fp32 router on the matrix pipe (csrc/gate.hip, gate_topk_f32_kernel): token counts
around its 16-token workgroups, the shortest and longest rows, few and many experts and
picks, ties, a NaN row; logits against float64 by a bound on their roundings."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("N,D,E,k", [
    (1, 64, 1, 1),        # one token, one chunk per wave, one expert
    (15, 384, 8, 2),
    (16, 384, 5, 3),      # a whole workgroup; experts that do not fill a lane group
    (17, 448, 16, 8),     # one token past it; both picks of a lane group; the longer form's shortest row
    (100, 768, 13, 6),
    (33, 1152, 8, 2),     # the longest row
])
@pytest.mark.parametrize("biased,renorm", [(False, False), (True, True)])
def test_fp32_router(N, D, E, k, biased, renorm):
    from dice_amd import ops
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(N + D)
    x, w = torch.randn(N, D, generator=g), torch.randn(E, D, generator=g) * 0.1
    if E >= 8:
        w[5] = w[2]                                   # ties: the lower id first
    bias = torch.randn(E, generator=g) if biased else None
    if biased and E >= 8:
        bias[5] = bias[2]
    idx, wt, logits, idx64 = ops.gate_topk(x.to(dev), w.to(dev), k, renorm, None if bias is None else bias.to(dev),
                                           want_logits=True, want_int64=True)
    idx, wt, logits = idx.cpu(), wt.cpu(), logits.cpu()
    assert torch.equal(idx64.cpu(), idx.long())
    want = x.double() @ w.double().T + (0 if bias is None else bias.double())
    # a sum of D / 64 products in chains, six pairwise additions and the bias, each rounded by 2^-24 of at most sum |x w|
    size = x.double().abs() @ w.double().abs().T + (0 if bias is None else bias.double().abs())
    assert bool(((logits.double() - want).abs() <= (D / 16 + 8) * 2.0 ** -24 * size).all())
    if E >= 8:
        assert torch.equal(logits[:, 5], logits[:, 2])
    # picks and weights follow from the returned logits
    p = torch.softmax(logits.double(), -1)
    order = torch.sort(p, dim=-1, descending=True, stable=True)
    # (scores of different logits may round alike: what is picked has the score, not always the id, of the sorted one)
    got = torch.gather(p, 1, idx.long())
    assert float((got - order.values[:, :k]).abs().max()) <= 2.0 ** -22
    if E >= 8:
        for row in idx.tolist():
            assert (5 not in row) or (2 in row and row.index(2) < row.index(5))
    ref = got / got.sum(-1, keepdim=True) if renorm and k > 1 else got
    assert float((wt.double() - ref).abs().max()) <= 2.0 ** -20   # exp, sums of 16, two divisions


def test_nan_row_stays_its_own():
    from dice_amd import ops
    dev = torch.device("cuda:0")
    g = torch.Generator().manual_seed(3)
    x, w = torch.randn(20, 384, generator=g), torch.randn(8, 384, generator=g) * 0.1
    clean = ops.gate_topk(x.to(dev), w.to(dev), 2)
    x[7, 100] = float("nan")
    x[18, 5] = float("inf")
    idx, wt = ops.gate_topk(x.to(dev), w.to(dev), 2)[:2]
    rows = [r for r in range(20) if r not in (7, 18)]
    assert torch.equal(idx[rows], clean[0][rows]) and torch.equal(wt[rows], clean[1][rows])
    assert bool(wt[7].isnan().all()) and bool(((idx >= 0) & (idx < 8)).all())
