"""Activation matrices of 2 GiB and more, where a descriptor of the gathering kernels ends:
rows on both sides of it, through both entry points of the grouped MLP (which know and do
not know the source's rows) and through the layer call, against float64."""
import pytest
import torch

from tests.helpers import check_rows

pytestmark = pytest.mark.gpu

GIB2 = 1 << 31
TOL = {torch.float32: 1e-5, torch.bfloat16: 1e-2, torch.float16: 2e-3}


@pytest.fixture(scope="module")
def dev():
    assert torch.cuda.is_available(), "these tests need the MI355X"
    from dice_amd import lib
    lib.load()
    return torch.device("cuda:0")


def _swiglu(x, w1, w2):
    inter = w2.shape[1]
    z = x.double() @ w1.double().t()
    return (torch.nn.functional.silu(z[:, :inter]) * z[:, inter:]) @ w2.double().t()


# rows per expert: few (the streaming kernels, fp32 the split ones) and many (the persistent ones)
@pytest.mark.parametrize("dtype,counts", [
    (torch.float32, [100, 0, 65, 1]),
    (torch.bfloat16, [100, 0, 65, 1]),
    (torch.float16, [700, 0, 330, 513]),
    (torch.bfloat16, [700, 0, 330, 513]),
])
@pytest.mark.parametrize("told", [True, False])
def test_grouped_rows_past_2gib(dev, dtype, counts, told):
    from dice_amd import lib, ops
    D, I, E, R, per = 512, 512, len(counts), sum(counts), 2
    g = torch.Generator(dev).manual_seed(R)
    rows = GIB2 // (D * dtype.itemsize) + 5000
    x = torch.empty(rows, D, dtype=dtype, device=dev)   # only the rows below are ever read
    inside = torch.randint(0, rows - 6000, (R,), generator=g, device=dev)
    past = torch.randint(rows - 5000, rows, (R,), generator=g, device=dev)
    edge = torch.tensor([rows - 5001, rows - 5000, 0, rows - 1], device=dev)   # the last row covered, the next one
    src = torch.where(torch.arange(R, device=dev) % 3 == 0, past, inside)
    src[:4] = edge
    x[src] = torch.randn(R, D, generator=g, device=dev).to(dtype)
    w1 = (torch.randn(E, 2 * I, D, generator=g, device=dev) * D ** -0.5).to(dtype)
    w2 = (torch.randn(E, D, I, generator=g, device=dev) * I ** -0.5).to(dtype)
    offsets = torch.tensor([0] + list(torch.tensor(counts).cumsum(0)), dtype=torch.int32, device=dev)
    perm = (src * per + 1).int()
    if told:
        out = ops.grouped_mlp(x, perm, per, offsets, R, w1, w2, "swiglu")
    else:
        h = torch.empty(R, I, dtype=dtype, device=dev)
        out = torch.empty(R, D, dtype=dtype, device=dev)
        lib.check(lib.load().dice_grouped_mlp(
            lib.ptr(x), lib.dtype_code(dtype), lib.ptr(perm), per, lib.ptr(offsets), E, R, D, I, lib.ptr(w1), None,
            lib.ptr(w2), None, None, None, lib.dtype_code(dtype), 0, lib.ptr(h), lib.ptr(out), 0, lib.stream_ptr()))
    o = 0
    for e, n in enumerate(counts):
        if n:
            check_rows(out[o:o + n], _swiglu(x[src[o:o + n]], w1[e], w2[e]), TOL[dtype], f"expert {e}")
        o += n


def test_layer_call_past_2gib(dev):
    """fp32 layer call whose input passes 2 GiB in its last rows."""
    from dice_amd import ParaMode, SparseMoeBlock
    D, E = 1024, 4
    N = GIB2 // (D * 4) + 3000
    g = torch.Generator(dev).manual_seed(3)
    with torch.device(dev):
        blk = SparseMoeBlock(D, 1, E, 1, pretraining_tp=1, layer_idx=0, total_layers=1, para_mode=ParaMode(),
                             variant="swiglu", n_shared_experts=None).eval()
    with torch.no_grad():
        for p in blk.parameters():
            p.copy_(torch.randn(p.shape, generator=g, device=dev) * p.shape[-1] ** -0.5)
    x = torch.randn(1, N, D, generator=g, device=dev)
    y = blk(x)[0]
    idx, wt = blk.gate(x)[:2]
    idx, wt = idx.view(-1), wt.view(-1).double()
    p = blk._packed
    pick = torch.cat([torch.arange(0, 100, device=dev), torch.arange(N - 3200, N, device=dev)])
    want = torch.empty(len(pick), D, dtype=torch.float64, device=dev)
    for e in range(E):
        here = idx[pick] == e
        want[here] = _swiglu(x[0, pick[here]], p.w1[e], p.w2[e]) * wt[pick[here], None]
    check_rows(y[pick], want, 1e-5, "rows around 2 GiB")
