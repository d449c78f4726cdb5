"""The fp32 expert GEMMs at the ends of the fp32 range: infinities, values that round to
infinity in bf16, NaN, and rows and weights too small for three bf16 parts."""
import pytest
import torch

from tests.test_gpu_split_f32 import dev  # noqa: F401

pytestmark = pytest.mark.gpu

INF, NAN, HUGE = float("inf"), float("nan"), 3.395e38   # (the largest bf16 number is 3.3895e38)


# (counts, D, I): the 64 x 64, 128 x 128, 256 x 256 and 256 x 128 tiles, see test_gpu_split_f32.py
SHAPES = [([63, 0, 64, 65], 128, 192), ([3001], 1536, 4096), ([8179], 768, 1024), ([8100, 0, 92], 2048, 256)]


def _problem(dev, counts, D, I, variant, seed):
    g = torch.Generator(dev).manual_seed(seed)
    E, R = len(counts), sum(counts)
    x = torch.randn(R, D, generator=g, device=dev)
    w1 = torch.randn(E, (2 if variant == "swiglu" else 1) * I, D, generator=g, device=dev) * D ** -0.5
    w2 = torch.randn(E, D, I, generator=g, device=dev) * I ** -0.5
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=dev)
    return x, w1, w2, offsets, R


def _run(x, w1, w2, offsets, R, variant, b1=None):
    from dice_amd import ops
    h = torch.empty(R, w2.shape[2], device=x.device)
    perm = torch.arange(R - 1, -1, -1, dtype=torch.int32, device=x.device)   # the source rows back to front
    return ops.grouped_mlp(x.flip(0).contiguous(), perm, 1, offsets, R, w1, w2, variant, b1, None, h=h), h


def _act(z, variant, I):
    if variant == "swiglu":
        return torch.nn.functional.silu(z[:, :I]) * z[:, I:]
    return torch.nn.functional.gelu(z, approximate="tanh")


def _same_kind(got, want):
    """Equal NaNs, equal infinities; what is finite is left to the caller."""
    want = want.float()
    assert torch.equal(got.isnan(), want.isnan())
    inf = want.isinf()
    assert torch.equal(got.isinf(), inf) and torch.equal(got[inf], want[inf])
    return ~(want.isnan() | inf)


@pytest.mark.parametrize("counts,D,I", SHAPES)
@pytest.mark.parametrize("variant", ["swiglu", "gelu_tanh"])
def test_infinities_and_nan(dev, counts, D, I, variant):
    x, w1, w2, offsets, R = _problem(dev, counts, D, I, variant, D)
    clean_out, clean_h = _run(x, w1, w2, offsets, R, variant)
    rows = {0: [(3, INF)], 5: [(D - 1, -INF)], 31: [(0, INF), (40, INF)], 40: [(17, NAN)], 62: [(9, HUGE)],
            R - 1: [(33, -HUGE), (34, HUGE)]}
    for r, put in rows.items():
        for c, v in put:
            x[r, c] = v
    out, h = _run(x, w1, w2, offsets, R, variant)
    special = torch.zeros(R, dtype=torch.bool, device=dev)
    special[list(rows)] = True
    assert torch.equal(out[~special], clean_out[~special]) and torch.equal(h[~special], clean_h[~special])
    for r in rows:
        e = int((offsets[1:] <= r).sum())
        z = x[r:r + 1].cpu().double() @ w1[e].cpu().double().t()
        want = _act(z, variant, I)
        fin = _same_kind(h[r:r + 1].cpu(), want)
        # sums of D products and an activation of slope 1.1 at most: D roundings of 2^-24 of sum |x w|, taken twice for SwiGLU
        if bool(fin.any()):
            size = (x[r:r + 1].cpu().double().abs() @ w1[e].cpu().double().abs().t())
            size = size[:, :I] * size[:, I:] if variant == "swiglu" else size
            err = (h[r:r + 1].cpu().double() - want).abs()
            assert bool((err <= 2.2 * (D + 8) * 2.0 ** -24 * size + 2.0 ** -149)[fin].all())
        _same_kind(out[r:r + 1].cpu(), h[r:r + 1].cpu().double() @ w2[e].cpu().double().t())


@pytest.mark.parametrize("counts,D,I", SHAPES)
def test_infinite_weight(dev, counts, D, I):
    x, w1, w2, offsets, R = _problem(dev, counts, D, I, "gelu_tanh", D + 1)
    clean_h = _run(x, w1, w2, offsets, R, "gelu_tanh")[1]
    w1[0, 5, 7] = INF
    x[2, 7] = 0.0                                     # 0 x infinity: NaN
    h = _run(x, w1, w2, offsets, R, "gelu_tanh")[1]
    n = counts[0]
    want = torch.where(x[:n, 7] > 0, INF, NAN)        # gelu(-infinity) is -infinity x 0
    assert torch.equal(h[:n, 5].isnan(), want.isnan()) and torch.equal(h[:n, 5].isinf(), want.isinf())
    same = torch.ones_like(h, dtype=torch.bool)
    same[:n, 5] = False
    same[2] = False
    assert torch.equal(h[same], clean_h[same])


@pytest.mark.parametrize("counts,D,I", SHAPES[:2])
@pytest.mark.parametrize("side", ["rows", "weights"])
@pytest.mark.parametrize("exponent", [-60, -70, -100, -112, -120])
def test_small_operands(dev, counts, D, I, side, exponent):
    """Rows and weights of magnitude 2^exponent: the error stays that of an fp32 sum of the same
    products (the third bf16 part of an operand below 2^-110 is out of range)."""
    x, w1, w2, offsets, R = _problem(dev, counts, D, I, "gelu_tanh", D + 2)
    if side == "rows":
        x[::3] *= 2.0 ** exponent
    else:
        w1[:, ::3] *= 2.0 ** exponent
    h = _run(x, w1, w2, offsets, R, "gelu_tanh")[1]
    o = 0
    for e, n in enumerate(counts):
        xe, we = x[o:o + n].double(), w1[e].double()
        err = (h[o:o + n].double() - _act(xe @ we.t(), "gelu_tanh", I)).abs()
        # (the products lie within 2^-149 of a multiple of it where they leave the normal range)
        assert bool((err <= 1.2 * (D + 8) * 2.0 ** -24 * (xe.abs() @ we.abs().t()) + D * 2.0 ** -149).all())
        o += n
