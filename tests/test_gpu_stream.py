"""The streaming expert GEMMs that small batches take (csrc/grouped_gemm_stream.hip):
row counts around the edges of their tiles, ragged and empty experts, fc2 whole and
cut along k, 16-bit and fp8 weights, against the oracle; and, where fc2 is not cut,
bit for bit against the persistent kernels (the sums are formed in the same order)."""
import contextlib

import pytest
import torch

from oracle import dice_oracle as O
from tests.helpers import block_from_params, check_rows

pytestmark = pytest.mark.gpu

TOL = {torch.bfloat16: 2e-2, torch.float16: 4e-3}
FP8_TOL = 5e-2


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from dice_amd import lib
    lib.load()
    return torch.device("cuda:0")


@contextlib.contextmanager
def hook(fc1):
    from dice_amd import lib
    lib.load().dice_set_gemm_config(fc1, 0)
    try:
        yield
    finally:
        lib.load().dice_set_gemm_config(0, 0)


def _params(D, E, k, ratio, variant, dtype, seed, skew=None):
    p = O.make_block_params(D, E, k, ratio, 2 if variant == "swiglu" else ratio, seed=seed, dtype=dtype, variant=variant,
                            gate_bias=skew)
    if variant == "gelu_tanh":
        g = torch.Generator().manual_seed(seed + 1)
        for e in list(p.experts) + [p.shared]:
            e.fc1_b = (torch.randn(e.fc1_b.shape, generator=g) * 0.1).to(dtype)
            e.fc2_b = (torch.randn(e.fc2_b.shape, generator=g) * 0.1).to(dtype)
    return p


# tokens: one expert takes them all where `E` is 1, so the row counts are exact there
@pytest.mark.parametrize("N,D,E,k,ratio,variant,dtype", [
    (1, 384, 4, 2, 4, "swiglu", torch.bfloat16),          # one row per tile
    (31, 128, 1, 1, 1, "swiglu", torch.bfloat16),         # less than a row block, one step of k per tile of fc2
    (128, 128, 1, 1, 2, "gelu_tanh", torch.float16),      # a whole 128-row tile
    (129, 320, 1, 1, 3, "swiglu", torch.float16),         # one row into the second; a partial weight tile
    (192, 192, 1, 1, 4, "gelu_tanh", torch.bfloat16),     # a whole 192-row tile
    (193, 256, 1, 1, 4, "swiglu", torch.bfloat16),        # one row past it
    (300, 1152, 8, 2, 4, "swiglu", torch.bfloat16),       # fc2 in two pieces (partial rows), shared fc2 whole
    (200, 1152, 8, 2, 4, "gelu_tanh", torch.float16),     # two pieces, shared fc2 (the longer one, first) too
    (100, 1152, 8, 4, 4, "swiglu", torch.bfloat16),       # the combine of four slots' partial rows
    (90, 1024, 4, 3, 4, "swiglu", torch.bfloat16),        # top-3: fc2 stays whole
    (257, 768, 33, 2, 4, "swiglu", torch.float16),        # many experts, some without rows
    (200, 1152, 17, 2, 4, "gelu_tanh", torch.bfloat16),   # fc2: routed tiles whole, the shared expert's cut
    (700, 1152, 8, 2, 4, "swiglu", torch.bfloat16),       # more fc2 tiles than compute units, 192-row tiles
    (40, 1152, 40, 2, 2, "swiglu", torch.float16),        # ... 128-row tiles, none cut
])
def test_block_on_the_streaming_kernels(dev, N, D, E, k, ratio, variant, dtype):
    skew = None if E < 8 else torch.linspace(2.0, -2.0, E)
    p = _params(D, E, k, ratio, variant, dtype, N, skew)
    x = torch.randn(1, N, D, generator=torch.Generator().manual_seed(N + 1)).to(dtype)
    blk = block_from_params(p, D, variant, dtype, dev)
    with hook(57):
        y = blk(x.to(dev))
        assert torch.equal(y, blk(x.to(dev)))
    want, _, _, logits = O.sparse_moe_block_forward(p, x)
    ok = ~O.gate_tie_rows(logits, k).view(-1)
    check_rows(y.cpu().view(-1, D)[ok], want.view(-1, D)[ok], TOL[dtype], "streaming kernels vs oracle")
    if variant == "swiglu" and D * ratio < 3456 and D >= 384:   # whole sums, no bias: the persistent kernels' bits
        with hook(56):
            assert torch.equal(y, blk(x.to(dev)))


@pytest.mark.parametrize("N,D,E,ratio,variant", [
    (40, 512, 4, 2, "swiglu"),        # 8 k steps of 64 and of 128 (fc2)
    (129, 1024, 4, 2, "gelu_tanh"),   # a second row tile; biases
    (300, 1152, 8, 4, "swiglu"),      # fc2 in two pieces
    (60, 1024, 20, 4, "gelu_tanh"),   # routed fc2 whole, the shared expert's cut
    (1500, 1024, 20, 4, "gelu_tanh"), # ... with more tiles than compute units
])
def test_fp8_weights_on_the_streaming_kernels(dev, N, D, E, ratio, variant):
    p = _params(D, E, 2, ratio, variant, torch.bfloat16, N)
    x = torch.randn(1, N, D, generator=torch.Generator().manual_seed(N + 1)).bfloat16()
    blk = block_from_params(p, D, variant, torch.bfloat16, dev)
    blk.quantize_fp8()
    with hook(57):
        y = blk(x.to(dev))
    with hook(56):
        other = blk(x.to(dev))
    want, _, _, logits = O.sparse_moe_block_forward(p, x)
    ok = ~O.gate_tie_rows(logits, 2).view(-1)
    check_rows(y.cpu().view(-1, D)[ok], want.view(-1, D)[ok], FP8_TOL, "fp8 weights vs bf16 masters")
    # (the persistent kernels on the same fp8 weights: outputs differ by roundings to bf16, 2^-9 each, of h and y)
    check_rows(y.cpu().view(-1, D), other.cpu().view(-1, D), 8e-3, "fp8 weights, streaming vs persistent")


@pytest.mark.parametrize("N", [320, 960, 961, 1920])
def test_put_and_skip_on_partial_rows(dev, N):
    """A put step writes the rows that its combine added up from pieces; a skip
    step, cut alike, reproduces the put step's output from them bit for bit.  From
    961 tokens on the put step takes the persistent kernels, whose rows are rounded
    before they are combined, and the skip step alone streams."""
    from dice_amd import lib
    D = 1152
    p = _params(D, 8, 2, 4, "swiglu", torch.bfloat16, 5)
    x = torch.randn(N, D, generator=torch.Generator().manual_seed(6)).bfloat16().to(dev)
    blk = block_from_params(p, D, "swiglu", torch.bfloat16, dev)
    mask = O.skip_mask(2 * N, "low").to(dev)
    cache = torch.empty_like(x)
    put = blk.run(x, lib.MODE_PUT, mask, None, cache).clone()
    assert torch.equal(put, blk.run(x))
    skip = blk.run(x, lib.MODE_SKIP, mask, cache, None)
    if N <= 960:
        assert torch.equal(put, skip)
    else:   # (a rounding of 2^-9 of the row that is not cached and one of the sum)
        check_rows(skip.cpu(), put.cpu(), 2.0 ** -8, "skip step on its own cache")


def test_entry_with_few_rows_in_a_large_batch(dev):
    """A lagged call whose entry holds few rows streams where its batch does not: the
    workspace, laid out for the batch, has no partial rows, so fc2 stays whole."""
    import ctypes
    from dice_amd import diep, lib
    D, E, N, R = 1152, 8, 3000, 64
    p = _params(D, E, 2, 4, "gelu_tanh", torch.bfloat16, 8)
    blk = block_from_params(p, D, "gelu_tanh", torch.bfloat16, dev)
    x = torch.randn(N, D, generator=torch.Generator().manual_seed(9)).bfloat16().to(dev)
    desc = blk._ensure(x)
    work = diep.LagEntry(x, E, 2, False, owner=blk)
    work.ensure_rows()
    work.x.copy_(x)
    work.offsets.copy_(torch.arange(E + 1, dtype=torch.int32) * (R // E))
    work.perm.zero_()
    work.perm[:R] = torch.arange(R, dtype=torch.int32, device=dev) * 2     # slot 0 of the first R tokens
    work.inv_perm.fill_(-1)
    work.inv_perm.view(-1, 2)[:R, 0] = torch.arange(R, dtype=torch.int32, device=dev)
    work.topk_weight.fill_(0.5)
    wd = work.desc()
    wd.max_rows = R

    def call():
        new = diep.LagEntry(x, E, 2, False, owner=blk)
        nd, y = new.desc(), torch.empty_like(x)
        ws = blk._workspace(desc, N, dev)
        lib.check(lib.load().dice_moe_forward_lagged(
            ctypes.byref(desc), ctypes.byref(desc), lib.ptr(x), N, 0, None, ctypes.byref(nd), ctypes.byref(wd), None,
            lib.MODE_PLAIN, None, None, 0, None, lib.ptr(y), None, None, lib.ptr(ws), ws.numel(), lib.stream_ptr()))
        return y

    y = call()
    with hook(56):
        want = call()
    # (sums of h and y in one order and bf16 roundings of 2^-9 each where a cut turn orders them otherwise)
    check_rows(y.cpu(), want.cpu(), 8e-3, "streaming vs persistent")
