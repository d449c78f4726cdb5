"""The persistent expert GEMMs whose operands are copied straight to LDS
(csrc/persist_dma.h) where they can go wrong: groups of 0 to 257 rows around the
edges of 16-row halves, 32- and 64-row blocks and 256-row tiles, the shortest
tile (six steps), weight tiles of 128, 192 and 256 rows, one that ends past the
matrix, with and without a bias, bf16 and fp16 - each stage against float64 of
the 16-bit operands it was given, element by element.  A launch of GROUPS gives a
workgroup one tile at most; MANY_GROUPS gives it three and more, of changing height,
so that copies cross into the next tile and the rows' numbers, the biases and the
scales staged a tile ahead change hands.

Bound: the fp32 sum of k products is off by at most k 2^-23 of the sum of the
products' magnitudes (a rounding to either side per addition), the activation
adds a few units of 2^-22 of its value, and the result is rounded to 16 bits
(half a unit in the last place: up to 2^-8 of a bf16 value, 2^-11 of an fp16 one, at
least 2^-25 there)."""
import pytest
import torch

from dice_amd import lib, ops

pytestmark = pytest.mark.gpu

GROUPS = [1, 16, 33, 63, 0, 257, 255, 640, 97, 15, 256, 130]
MANY_GROUPS = [67 * e % 401 for e in range(48)]   # 0 .. 400 rows in no order: tiles with one to four live 64-row blocks
HALF_ULP = {torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}   # of a value just above a power of two


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    lib.load()
    return torch.device("cuda:0")


def _check(got, want, magnitude, dtype, k, what):
    bound = HALF_ULP[dtype] * want.abs() * 1.01 + k * 2.0 ** -23 * magnitude + 2.0 ** -25
    over = (got.double() - want).abs() / bound
    assert torch.isfinite(got.float()).all(), what
    assert float(over.max()) <= 1.0, f"{what}: {float(over.max()):.2f} x the bound at {int(over.argmax())}"


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("variant,D,inter,slim", [
    ("swiglu", 384, 768, False),      # fc2 on 192 weight rows
    ("swiglu", 640, 768, False),      # ... on 256, the last tile half past the matrix
    ("swiglu", 384, 1024, True),      # 128 weight rows in both stages
    ("gelu_tanh", 384, 1024, False),  # bias: fc1 on 256, fc2 on 192
    ("gelu_tanh", 384, 1024, True),   # ... fc2 on 128
])
def test_ragged_groups_against_float64(dev, variant, D, inter, slim, dtype):
    _both_stages_against_float64(dev, GROUPS, variant, D, inter, slim, dtype)


def _turns(groups, outputs, per_tile):
    """Tiles of the fullest workgroup, at least, where a tile has `per_tile` of the `outputs` columns."""
    tiles = sum(-(-g // 256) for g in groups) * -(-outputs // per_tile)
    return -(-tiles // torch.cuda.get_device_properties(0).multi_processor_count)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("variant,D,inter,slim,stage,per_tile", [
    ("swiglu", 384, 2048, False, 1, 128),      # fc1 in tiles of six steps, its rows through the row table
    ("swiglu", 384, 1024, True, 1, 64),        # ... on 128 weight rows
    ("swiglu", 2688, 384, False, 2, 192),      # fc2 in tiles of six steps, on 192 weight rows
    ("swiglu", 3200, 384, False, 2, 256),      # ... on 256, the last tile half past the matrix
    ("swiglu", 1920, 384, True, 2, 128),       # ... on 128
    ("gelu_tanh", 384, 3072, False, 1, 256),   # fc1 with a bias and the row table
    ("gelu_tanh", 2688, 512, False, 2, 192),   # fc2 with a bias, on 192
    ("gelu_tanh", 1920, 512, True, 2, 128),    # ... on 128
])
def test_tile_switches_on_ragged_groups_against_float64(dev, variant, D, inter, slim, stage, per_tile, dtype):
    assert _turns(MANY_GROUPS, inter if stage == 1 else D, per_tile) >= 3
    _both_stages_against_float64(dev, MANY_GROUPS, variant, D, inter, slim, dtype)


@pytest.mark.parametrize("h_blocks", [False, True])
@pytest.mark.parametrize("variant", ["swiglu", "gelu_tanh"])
@pytest.mark.parametrize("D,inter", [(768, 3072), (3072, 768)])   # fc1 / fc2 in tiles of six steps
def test_fp8_tile_switches_give_the_bits_of_a_launch_per_group(dev, variant, D, inter, h_blocks):
    """e4m3 rows: a launch of all groups against one launch per group, in which no workgroup has a
    second tile (tests/test_gpu_fp8_act.py holds such launches against the oracle).  A row's sums run over the
    same products in the same order in both: the same bytes, of h and its block scales as well."""
    groups, k = [g for g in MANY_GROUPS if g], 2
    widths = {"swiglu": (128, 256), "gelu_tanh": (256, 256)}[variant]
    assert _turns(groups, *((inter, widths[0]) if D < inter else (D, widths[1]))) >= 3
    assert _turns([max(groups)], inter, widths[0]) == _turns([max(groups)], D, widths[1]) == 1
    gen = torch.Generator(dev).manual_seed(15)
    E, rows = len(groups), sum(groups)

    def normal(*shape, std):
        return torch.randn(*shape, generator=gen, device=dev).mul_(std)

    x = normal((rows + k - 1) // k, D, std=1.0).bfloat16()
    w1, s1 = ops.quantize_fp8_rowwise(normal(E, (2 if variant == "swiglu" else 1) * inter, D, std=D ** -0.5).bfloat16())
    w2, s2 = ops.quantize_fp8_rowwise(normal(E, D, inter, std=inter ** -0.5).bfloat16())
    b1 = b2 = None
    if variant == "gelu_tanh":
        b1, b2 = normal(E, inter, std=1.0), normal(E, D, std=1.0)
    perm = torch.randperm(x.shape[0] * k, generator=torch.Generator().manual_seed(16))[:rows].to(dev, torch.int32)
    ends = torch.tensor([0] + groups).cumsum(0).to(dev, torch.int32)

    def mlp(lo, hi, first, last):
        some = slice(first, last)
        out, h = ops.grouped_mlp_a8(
            x, perm[lo:hi].clone(), k, ends[first:last + 1] - ends[first], hi - lo, w1[some], w2[some],
            s1[some], s2[some], variant, None if b1 is None else b1[some], None if b2 is None else b2[some],
            h=torch.zeros((hi - lo + 2, inter), dtype=torch.bfloat16, device=dev), h_blocks=h_blocks)
        return (out,) + (ops.split_h_blocks(h, hi - lo, inter) if h_blocks else (h[:hi - lo],))

    whole = mlp(0, rows, 0, E)
    assert torch.isfinite(whole[0].float()).all()
    for e in range(E):
        lo, hi = int(ends[e]), int(ends[e + 1])
        for name, got, want in zip(("out", "h", "exponents of h"), whole, mlp(lo, hi, e, e + 1)):
            assert torch.equal(got[lo:hi].view(torch.uint8), want.contiguous().view(torch.uint8)), f"{name} of expert {e}, {hi - lo} rows"


def _both_stages_against_float64(dev, groups, variant, D, inter, slim, dtype):
    gen = torch.Generator(dev).manual_seed(5)
    E, rows, k = len(groups), sum(groups), 2
    assert rows > 128 * E                     # (fewer rows per expert would take other kernels)

    def normal(*shape, std):
        return torch.randn(*shape, generator=gen, device=dev).mul_(std).to(dtype)

    up = 2 if variant == "swiglu" else 1
    n_src = (rows + k - 1) // k
    x, w1, w2 = normal(n_src, D, std=1.0), normal(E, up * inter, D, std=D ** -0.5), normal(E, D, inter, std=inter ** -0.5)
    b1 = b2 = None
    if variant == "gelu_tanh":
        b1, b2 = (torch.randn(E, n, generator=gen, device=dev) for n in (inter, D))
    perm = torch.randperm(n_src * k, generator=torch.Generator().manual_seed(6))[:rows].to(dev, torch.int32)
    offsets = torch.tensor([sum(groups[:e]) for e in range(E + 1)], device=dev, dtype=torch.int32)
    guard = 7.0                               # rows past the groups' end stay as they are
    h = torch.full((rows + 3, inter), guard, device=dev, dtype=dtype)
    out = torch.full((rows + 3, D), guard, device=dev, dtype=dtype)
    # 21: the persistent kernels, 54: ... on 128 weight rows
    lib.load().dice_set_gemm_config(54 if slim and variant == "swiglu" else 21, 54 if slim else 21)
    try:
        ops.grouped_mlp(x, perm, k, offsets, rows, w1, w2, variant, b1, b2, h=h, out=out)
    finally:
        lib.load().dice_set_gemm_config(0, 0)
    assert bool((h[rows:] == guard).all()) and bool((out[rows:] == guard).all())
    src = x.double()[(perm // k).long()]
    for e in range(E):
        lo, hi = int(offsets[e]), int(offsets[e + 1])
        if lo == hi:
            continue
        a = src[lo:hi]
        s, mag = a @ w1[e].double().t(), a.abs() @ w1[e].double().abs().t()
        if variant == "swiglu":
            g, u = s[:, :inter], s[:, inter:]
            want = torch.nn.functional.silu(g) * u
            # (silu's slope is at most 1.1)
            m = mag[:, :inter] * 1.1 * u.abs() + torch.nn.functional.silu(g).abs() * mag[:, inter:] + want.abs()
        else:
            s, mag = s + b1[e].double(), mag + b1[e].double().abs()
            want, m = torch.nn.functional.gelu(s, approximate="tanh"), 1.13 * mag + s.abs()
        _check(h[lo:hi], want, m, dtype, D, f"fc1 of expert {e}, {hi - lo} rows")
        hh = h[lo:hi].double()
        want, m = hh @ w2[e].double().t(), hh.abs() @ w2[e].double().abs().t()
        if b2 is not None:
            want, m = want + b2[e].double(), m + b2[e].double().abs()
        _check(out[lo:hi], want, m, dtype, inter, f"fc2 of expert {e}, {hi - lo} rows")
