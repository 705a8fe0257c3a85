"""Weight- and bias-gradient kernel against fp64 products of the same 16-bit operands."""
import pytest
import torch

from sparseattention_amd import _lib
from sparseattention_amd.ops.linear import linear, query_key_value_rows

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _close(got, ref, rows, eps, what):
    # fp32 sum of `rows` products of size 1: partial sums of size sqrt(k), each rounded to 2^-24, signs
    # independent, so sigma < rows * 2^-24; the result rounded once to its type
    err = (got.double().cpu() - ref).abs()
    assert bool((err <= 4 * (rows + 8) * 2.0 ** -24 + eps * ref.abs()).all()), "%s: %.3e" % (what, float(err.max()))


# (rows, O, I): one row, less / more than a stage of 64 rows, the chunk's edge (128), a partly filled tile
# on either side, several tiles and chunks, a single tile with many chunks
@pytest.mark.parametrize("shape", [(1, 8, 8), (63, 128, 128), (65, 136, 64), (128, 64, 200), (129, 256, 128), (1000, 384, 264),
                                   (4095, 512, 512), (20000, 128, 128), (3000, 2304, 768)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("wide", [True, False])
def test_weight_grad(shape, dtype, wide):
    rows, O, I = shape
    g = torch.Generator().manual_seed(rows + O)
    # operands that are column slices of wider matrices
    dy = torch.randn(rows, O + 16, generator=g).to(dtype)[:, 8:8 + O]
    x = torch.randn(rows, I + 8, generator=g).to(dtype)[:, :I]
    dyd = torch.empty(rows, O + 16, dtype=dtype, device=DEV)[:, 8:8 + O].copy_(dy)
    xd = torch.empty(rows, I + 8, dtype=dtype, device=DEV)[:, :I].copy_(x)
    out = torch.float32 if wide else dtype
    r = _lib.ext().weight_grad([(dyd, xd, 0)], O, out, True)
    assert r is not None and r[0].dtype == out and r[0].shape == (O, I) and r[1].shape == (O,)
    # rounding to 8 / 11 significant bits: half a unit of the last, relative to the smallest value with it
    eps = 0.0 if wide else {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[dtype]
    _close(r[0], dy.double().t() @ x.double(), rows, eps, "dw")
    _close(r[1], dy.double().sum(0), rows, eps, "db")
    assert torch.equal(r[0], _lib.ext().weight_grad([(dyd, xd, 0)], O, out, False)[0])


def test_weight_grad_segments():
    """Three pairs adding up, two of them on the lower rows of the result; rows without any are zero."""
    D, g = 96, torch.Generator().manual_seed(3)
    mk = lambda r, c: torch.randn(r, c, generator=g).to(torch.bfloat16)
    pairs = [(mk(500, 3 * D), mk(500, D), 0), (mk(700, 2 * D), mk(700, D), D), (mk(3, 2 * D), mk(3, D), D)]
    got, _ = _lib.ext().weight_grad([(a.to(DEV), b.to(DEV), f) for a, b, f in pairs], 3 * D + 8, torch.float32, False)
    want = torch.zeros(3 * D + 8, D, dtype=torch.float64)
    for a, b, f in pairs:
        want[f:f + a.shape[1]] += a.double().t() @ b.double()
    _close(got, want, 1203, 0.0, "dw")


def test_weight_grad_keeps_infinities_out_of_other_rows():
    """Rows behind the last one take no part, whatever the last row holds."""
    dy, x = torch.ones(70, 16, device=DEV, dtype=torch.float16), torch.ones(70, 16, device=DEV, dtype=torch.float16)
    x[69, 3] = float("inf")
    dw, db = _lib.ext().weight_grad([(dy, x, 0)], 16, torch.float32, True)
    assert torch.isinf(dw[:, 3]).all() and torch.isfinite(dw[:, [0, 1, 2] + list(range(4, 16))]).all()
    assert bool((dw[:, 0] == 70).all()) and bool((db == 70).all())


def test_weight_grad_refuses():
    f = _lib.ext().weight_grad
    a, b = torch.zeros(64, 24, device=DEV, dtype=torch.float16), torch.zeros(64, 16, device=DEV, dtype=torch.float16)
    assert f([(a, b, 0)], 24, torch.float32, True) is not None
    assert f([(a[:, :20], b, 0)], 20, torch.float32, False) is None          # 20 columns
    assert f([(a[:, 4:20], b, 0)], 16, torch.float32, False) is None         # rows off by 8 bytes
    assert f([(a, b.float(), 0)], 24, torch.float32, False) is None          # types differ
    assert f([(a.float(), b.float(), 0)], 24, torch.float32, False) is None  # fp32 operands
    assert f([(a, b, 0)], 24, torch.bfloat16, False) is None
    assert f([(a, b, 0), (a, b, 0)], 24, torch.float32, True) is None        # a bias goes with one pair
    assert f([(a[:63], b, 0)], 24, torch.float32, False) is None


# ---------------------------------------------------------------- the layer that uses it
def _layers(dtype, bias, O=96, I=64):
    torch.manual_seed(1)
    layer = torch.nn.Linear(I, O, bias=bias).to(DEV).to(dtype)
    ref = torch.nn.Linear(I, O, bias=bias).double()
    ref.load_state_dict({k: v.double().cpu() for k, v in layer.state_dict().items()})
    return layer, ref


@pytest.mark.parametrize("bias", [True, False])
@pytest.mark.parametrize("amp", [None, torch.float16, torch.bfloat16])
@pytest.mark.parametrize("view", [False, True])
def test_linear_against_fp64(bias, amp, view):
    dtype = torch.float32 if amp else torch.bfloat16
    low = amp or dtype
    layer, ref = _layers(dtype, bias)
    g = torch.Generator().manual_seed(2)
    x = torch.randn(3, 50, 64, generator=g).to(low).to(dtype)
    dy = torch.randn(3, 50, 96, generator=g).to(low)
    xd = x.to(DEV).transpose(0, 1).contiguous().transpose(0, 1) if view else x.to(DEV)
    xd.requires_grad_(True)
    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        y = linear(layer, xd)
        assert "Linear" in y.grad_fn.name() and y.grad_fn.name() != torch.nn.functional.linear(xd, layer.weight).grad_fn.name()
        want = layer(xd.detach())
    assert torch.equal(y, want) and y.dtype == low
    y.backward(dy.to(DEV))
    # the reference on the operands as rounded to the 16-bit type
    with torch.no_grad():
        ref.weight.copy_(layer.weight.to(low).double().cpu())
    xr = x.double().requires_grad_(True)
    ref(xr).backward(dy.double())
    half = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}
    _close(layer.weight.grad, ref.weight.grad, 150, 0.0 if amp else half[low], "dw")
    if bias:
        _close(layer.bias.grad, ref.bias.grad, 150, 0.0 if amp else half[low], "db")
    _close(xd.grad, xr.grad, 96, half[low], "dx")


def test_linear_leaves_other_calls_to_the_layer():
    layer, _ = _layers(torch.bfloat16, True)
    x = torch.randn(5, 64, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        assert torch.equal(linear(layer, x), layer(x))
    seen = []
    h = layer.register_forward_hook(lambda m, a, o: seen.append(1))
    linear(layer, x)
    assert seen == [1]
    h.remove()
    wide = torch.nn.Linear(64, 20).to(DEV).to(torch.bfloat16)  # 20 outputs: no whole 16-byte pieces
    linear(wide, x).sum().backward()
    assert wide.weight.grad is not None

    class Net(torch.nn.Module):
        def __init__(self):
            super().__init__()
            self.layer = layer

        def forward(self, t):
            return linear(self.layer, t)

    traced = torch.jit.trace(Net(), x, check_trace=False)
    assert torch.equal(traced(2 * x), layer(2 * x))
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(x, torch.ones_like(x))
        t = torch.autograd.forward_ad.unpack_dual(linear(layer, d)).tangent
    assert torch.equal(t, torch.nn.functional.linear(torch.ones_like(x), layer.weight))


def test_linear_differentiated_twice():
    layer, _ = _layers(torch.bfloat16, False)
    x = torch.randn(40, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True)

    def second(f):
        gx, gw = torch.autograd.grad(f(x).square().sum(), [x, layer.weight], create_graph=True)
        return torch.autograd.grad(gx.square().sum() + gw.float().square().sum(), [x, layer.weight])

    for a, b in zip(second(lambda t: linear(layer, t)), second(layer)):
        assert torch.equal(a, b)


# ------------------------------------------------------- queries, keys and values of leaves and nodes
@pytest.mark.parametrize("shape", [(1, 1, 1, 8), (2, 64, 63, 96), (3, 5, 9, 264), (1, 2000, 1999, 64)])
@pytest.mark.parametrize("types", [(None, torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32, torch.float16),
                                   (torch.bfloat16, torch.float32, torch.float32), (torch.float16, torch.float16, torch.float32)])
def test_query_key_value_rows(shape, types):
    B, N, M, C = shape
    amp, xt, yt = types
    low = amp or xt
    wt = torch.float32 if amp else low
    g = torch.Generator().manual_seed(C)
    mk = lambda *s: torch.randn(*s, generator=g).to(low)
    x, y, gq, gk, gv = mk(B, N, C).to(xt), mk(B, M, C).to(yt), mk(B, N, C), mk(B, N + M, C), mk(B, N + M, C)
    lq, lk, lv = (torch.nn.Linear(C, C, bias=False).to(DEV).to(wt) for _ in range(3))
    xd, yd = x.to(DEV).requires_grad_(True), y.to(DEV).requires_grad_(True)
    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        q, k, v = query_key_value_rows(lq, lk, lv, xd, yd)
        xs = xd.detach().to(low)
        xy = torch.cat([xs, yd.detach().to(low)], dim=1)
        assert k.dtype == low and torch.equal(q, lq(xs)) and torch.equal(k, lk(xy)) and torch.equal(v, lv(xy))
    torch.autograd.backward([q, k, v], [gq.to(DEV), gk.to(DEV), gv.to(DEV)])
    # what the library's products give, added in fp32 and rounded to the inputs' types
    back = lambda go, layer: go.to(DEV).view(-1, C).mm(layer.weight.detach().to(low)).float().view(B, -1, C)
    d = back(gk, lk) + back(gv, lv)
    assert torch.equal(xd.grad, (d[:, :N] + back(gq, lq)).to(xt)) and torch.equal(yd.grad, d[:, N:].to(yt))
    half = 0.0 if amp else {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[low]
    for layer, go, rows in ((lq, gq, xs), (lk, gk, xy), (lv, gv, xy)):
        want = go.double().view(-1, C).t() @ rows.double().cpu().reshape(-1, C)
        _close(layer.weight.grad, want, B * (N + M), half, "dw")


def test_query_key_value_rows_partial_use():
    """Some results unused, only one input needing a gradient, layers with hooks or biases left alone."""
    lq, lk, lv = (torch.nn.Linear(64, 64, bias=False).to(DEV).to(torch.bfloat16) for _ in range(3))
    x = torch.randn(2, 8, 64, device=DEV, dtype=torch.bfloat16)
    y = torch.randn(2, 7, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    q, k, v = query_key_value_rows(lq, lk, lv, x, y)
    v.sum().backward()
    assert lk.weight.grad is None and lq.weight.grad is None and lv.weight.grad is not None
    assert torch.equal(y.grad, torch.ones_like(v.detach()).matmul(lv.weight.detach())[:, 8:])
    y.grad = None
    q, k, v = query_key_value_rows(lq, lk, lv, x, y)
    ((k + v).sum() + q.sum()).backward()
    assert y.grad is not None and x.grad is None and lq.weight.grad is not None
    x.requires_grad_(True)
    query_key_value_rows(lq, lk, lv, x, y)[0].sum().backward()
    assert torch.equal(x.grad, torch.ones_like(x).matmul(lq.weight.detach()))
    with torch.no_grad():
        assert query_key_value_rows(lq, lk, lv, x, y) is None
    assert query_key_value_rows(lq, torch.nn.Linear(64, 64).to(DEV).to(torch.bfloat16), lv, x, y) is None
    assert query_key_value_rows(lq, lk, lv, x.float(), y.float()) is None


def test_query_key_value_rows_differentiated_twice():
    lq, lk, lv = (torch.nn.Linear(32, 32, bias=False).to(DEV).to(torch.bfloat16) for _ in range(3))
    x, y = (torch.randn(2, n, 32, device=DEV, dtype=torch.bfloat16, requires_grad=True) for n in (8, 7))

    def second(f):
        q, k, v = f()
        gx, gw = torch.autograd.grad(q.float().square().sum() + (k * v).float().sum(), [x, lk.weight], create_graph=True)
        return torch.autograd.grad(gx.float().square().sum() + gw.float().square().sum(), [x, y, lq.weight, lv.weight])

    def plain():
        xy = torch.cat([x, y], dim=1)
        return lq(x), lk(xy), lv(xy)

    for a, b in zip(second(lambda: query_key_value_rows(lq, lk, lv, x, y)), second(plain)):
        # bf16 through two backward passes, summed in other orders: a few units of 2^-8 of the norm
        assert (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
