"""Weight- and bias-gradient kernel against fp64 products of the same 16-bit operands."""
import pytest
import torch

from sparseattention_amd import _lib
from sparseattention_amd.ops.linear import key_value_rows, linear

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


# ---------------------------------------------------------------- keys and values of leaves and nodes
@pytest.mark.parametrize("shape", [(1, 1, 1, 8), (2, 64, 63, 96), (3, 5, 9, 264), (1, 2000, 1999, 64)])
@pytest.mark.parametrize("types", [(None, torch.bfloat16, torch.bfloat16), (torch.float16, torch.float32, torch.float16),
                                   (torch.bfloat16, torch.float32, torch.float32), (torch.float16, torch.float16, torch.float32)])
def test_key_value_rows(shape, types):
    B, N, M, C = shape
    amp, xt, yt = types
    low = amp or xt
    wt = torch.float32 if amp else low
    g = torch.Generator().manual_seed(C)
    mk = lambda *s: torch.randn(*s, generator=g).to(low)
    x, y, gk, gv = mk(B, N, C).to(xt), mk(B, M, C).to(yt), mk(B, N + M, C), mk(B, N + M, C)
    lk, lv = (torch.nn.Linear(C, C, bias=False).to(DEV).to(wt) for _ in range(2))
    xd, yd = x.to(DEV).requires_grad_(True), y.to(DEV).requires_grad_(True)
    with torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        k, v = key_value_rows(lk, lv, xd, yd)
        xy = torch.cat([xd.detach().to(low), yd.detach().to(low)], dim=1)
        assert k.dtype == low and torch.equal(k, lk(xy)) and torch.equal(v, lv(xy))
    torch.autograd.backward([k, v], [gk.to(DEV), gv.to(DEV)])
    # what the library's products give, added in fp32 and rounded to the inputs' types
    d = gk.to(DEV).view(-1, C).mm(lk.weight.detach().to(low)).float() + gv.to(DEV).view(-1, C).mm(lv.weight.detach().to(low)).float()
    d = d.view(B, N + M, C)
    assert torch.equal(xd.grad, d[:, :N].to(xt)) and torch.equal(yd.grad, d[:, N:].to(yt))
    half = 0.0 if amp else {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[low]
    for layer, go in ((lk, gk), (lv, gv)):
        want = go.double().view(-1, C).t() @ xy.double().cpu().view(-1, C)
        _close(layer.weight.grad, want, B * (N + M), half, "dw")


def test_key_value_rows_partial_use():
    """Only one result used, only one input needing a gradient, layers with hooks or biases left alone."""
    lk, lv = (torch.nn.Linear(64, 64, bias=False).to(DEV).to(torch.bfloat16) for _ in range(2))
    x = torch.randn(2, 8, 64, device=DEV, dtype=torch.bfloat16)
    y = torch.randn(2, 7, 64, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    k, v = key_value_rows(lk, lv, x, y)
    v.sum().backward()
    assert lk.weight.grad is None and lv.weight.grad is not None
    want = torch.ones_like(v.detach()).matmul(lv.weight.detach())[:, 8:]
    assert torch.equal(y.grad, want)
    y.grad = None
    k, v = key_value_rows(lk, lv, x, y)
    (k + v).sum().backward()
    assert y.grad is not None and x.grad is None
    with torch.no_grad():
        assert key_value_rows(lk, lv, x, y) is None
    assert key_value_rows(torch.nn.Linear(64, 64).to(DEV).to(torch.bfloat16), lv, x, y) is None
    assert key_value_rows(lk, lv, x.float(), y.float()) is None
