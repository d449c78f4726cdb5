"""The fp32 expert GEMMs on the bf16 matrix pipe (csrc/grouped_gemm_split.hip): every
tile shape at ragged row counts, empty experts, slot-order and grouped output, against
float64; whole and cut fc2 of the layer call against each other."""
import pytest
import torch

from oracle import dice_oracle as O
from tests.helpers import block_from_params

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from dice_amd import lib
    lib.load()
    return torch.device("cuda:0")


def _sum_error(k):
    """Relative l2 error of sums of k products: six roundings per sixteen products, each at most
    2^-24 of a running sum that is on average no larger than the final one, independent."""
    return 2.0 ** -24 * (6 * k / 16) ** 0.5


def _rel(got, want):
    return float((got.double() - want).norm() / want.norm())


# rows per expert; the comments name the tiles that the two stages take
@pytest.mark.parametrize("counts,D,I,variant", [
    ([1], 64, 64, "swiglu"),                            # 64 x 64; one row, two lines of k
    ([63, 0, 64, 65], 128, 192, "gelu_tanh"),           # 64 x 64; around a tile, an expert without rows
    ([31, 33, 129, 0, 0, 7], 384, 1536, "swiglu"),      # 64 x 64
    ([3001], 1536, 4096, "gelu_tanh"),                  # 128 x 128
    ([8179], 768, 1024, "swiglu"),                      # 256 x 256, 256 x 128
    ([8100, 0, 92], 2048, 256, "gelu_tanh"),            # 64 x 64, 256 x 256
])
def test_against_float64(dev, counts, D, I, variant):
    from dice_amd import ops
    g = torch.Generator(dev).manual_seed(sum(counts) + D)
    E, R = len(counts), sum(counts)
    swiglu = variant == "swiglu"
    x = torch.randn(R, D, generator=g, device=dev)
    w1 = torch.randn(E, (2 if swiglu else 1) * I, D, generator=g, device=dev) * D ** -0.5
    w2 = torch.randn(E, D, I, generator=g, device=dev) * I ** -0.5
    b1 = None if swiglu else torch.randn(E, I, generator=g, device=dev) * 0.1
    b2 = None if swiglu else torch.randn(E, D, generator=g, device=dev) * 0.1
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=dev)
    perm = torch.randperm(R, generator=g, device=dev).int()
    h = torch.full((R, I), float("nan"), device=dev)
    out = ops.grouped_mlp(x, perm, 1, offsets, R, w1, w2, variant, b1, b2, h=h)
    by_slot = ops.grouped_mlp(x, perm, 1, offsets, R, w1, w2, variant, b1, b2, scatter_to_slots=True, n_out_rows=R)
    assert torch.equal(by_slot[perm.long()], out)
    o = 0
    for e, n in enumerate(counts):
        if n == 0:
            continue
        rows = slice(o, o + n)
        z = x[perm[rows].long()].double() @ w1[e].double().t()
        if swiglu:
            want = torch.nn.functional.silu(z[:, :I]) * z[:, I:]
        else:
            want = torch.nn.functional.gelu(z + b1[e].double(), approximate="tanh")
        # two sums, a slope of at most 1.1 each, and four ulps for the exponential, the reciprocal and the products
        assert _rel(h[rows], want) < 2.2 * _sum_error(D) + 2.0 ** -21
        want = h[rows].double() @ w2[e].double().t() + (0 if b2 is None else b2[e].double())
        assert _rel(out[rows], want) < _sum_error(I) + 2.0 ** -24
        o += n


@pytest.mark.parametrize("N,D,E,k,ratio", [
    (33, 384, 8, 2, 4),      # routed fc2 in three pieces, shared in two
    (130, 768, 8, 1, 4),     # four pieces, one slot per token
    (65, 512, 4, 4, 4),      # four slots
    (64, 384, 8, 3, 4),      # top-3: fc2 stays whole
])
def test_layer_with_cut_fc2(dev, N, D, E, k, ratio):
    from dice_amd import lib
    p = O.make_block_params(D, E, k, ratio, 2, seed=N, dtype=torch.float32)
    x = torch.randn(N, D, generator=torch.Generator().manual_seed(N)).to(dev)
    blk = block_from_params(p, D, "swiglu", torch.float32, dev)
    y = blk.run(x).clone()
    assert torch.equal(y, blk.run(x))
    whole = block_from_params(p, D, "swiglu", torch.float32, dev)
    whole.batch_invariant = True   # (never cut)
    # two fc2 sums, formed in another order each
    assert _rel(y, whole.run(x).double()) < 2 * _sum_error(D * ratio)
    if k == 2:
        mask = O.skip_mask(k * N, "low").to(dev)
        cache = torch.empty_like(x)
        assert torch.equal(y, blk.run(x, lib.MODE_PUT, mask, None, cache))
        assert torch.equal(y, blk.run(x, lib.MODE_SKIP, mask, cache, None))


def _parts(v):
    a = v.bfloat16().float()
    b = (v - a).bfloat16().float()
    return a.double(), b.double(), (v - a - b).double()


@pytest.mark.parametrize("products", [1, 2])
def test_sums_of_few_products(dev, products):
    """Where nothing averages out: one or two products that are not zero.  The parts left out are at most 2^-24 of a
    product.  An addition of the matrix pipe is good to an ulp of its sum (2^-23): the last of the first product's six
    (those before it act on sums of at most 2^-6), all six of the second's."""
    from dice_amd import lib
    K, N, R = 512, 256, 300
    g = torch.Generator().manual_seed(products)
    v = 1 + torch.rand(R, generator=g)
    v[:8] = 1.0038986   # (next to the worst pair: parts of 2^-8 and 2^-17)
    h = torch.zeros(R, K)
    at = torch.randint(0, K // products, (R,), generator=g)
    for i in range(products):
        h[torch.arange(R), at + i * (K // products)] = v.roll(i)
    w = (1 + torch.rand(N, K, generator=g)) * (1 - 2 * (torch.rand(N, K, generator=g) < 0.5).float())
    w[:16] = 1.0038986
    # the parts themselves
    a, b, c = _parts(torch.cat([v, w.reshape(-1)]))
    whole = torch.cat([v, w.reshape(-1)]).double()
    assert torch.equal(a + b + c, whole) and torch.equal(c, c.float().bfloat16().double())
    lost = 2 * b.abs() * c.abs() + c * c
    assert float((lost / (whole * whole)).max()) <= 2.0 ** -24 * (1 + 2.0 ** -8)
    out = torch.empty(R, N, device=dev)
    hd, wd, off = h.to(dev), w.to(dev), torch.tensor([0, R], dtype=torch.int32, device=dev)
    p = lib.ptr
    lib.check(lib.load().dice_grouped_mlp_rows(2, p(hd), R, 0, None, 1, p(off), 1, R, N, K, p(wd), None, p(wd), None,
                                               None, None, 0, 0, p(hd), p(out), 0, lib.stream_ptr()))
    want, size = h.double() @ w.double().t(), h.double() @ w.double().abs().t()
    bound = 2.0 ** -24 * (1 + 2 * (1 + 6 * (products - 1)) + 2.0 ** -3) * size
    assert bool(((out.cpu().double() - want).abs() <= bound).all())
