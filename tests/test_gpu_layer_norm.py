"""Residual sum + layer norm kernel against torch's layer norm in fp64 on the same inputs."""
import pytest
import torch
import torch.nn.functional as F

from sparseattention_amd import _lib
from sparseattention_amd.transformer import add_layer_norm, layer_norm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# (rows, channels): one row, more rows than resident row groups, half-wavefront rows, partly filled last
# pieces, the widest row of each piece count
@pytest.mark.parametrize("shape", [(1, 8), (3, 24), (5, 256), (700, 320), (9001, 512), (130, 768), (33, 1000), (17, 1536), (40, 2048)])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("add", [True, False])
def test_add_layer_norm(shape, dtype, add):
    rows, C = shape
    if C * torch.finfo(dtype).bits > 16 * 2048:
        C //= 2
    g = torch.Generator().manual_seed(rows + C)
    mk = lambda *s: torch.randn(*s, generator=g).to(dtype)
    a, b, w, be, dn, ds = mk(rows, C) + 1, mk(rows, C), mk(C), mk(C), mk(rows, C), mk(rows, C)
    norm = torch.nn.LayerNorm(C).to(DEV).to(dtype)
    with torch.no_grad():
        norm.weight.copy_(w)
        norm.bias.copy_(be)
    ad, bd = a.to(DEV).requires_grad_(True), b.to(DEV).requires_grad_(True)
    # the reference on the sum as rounded to the element type
    s = ((a + b) if add else a).double().requires_grad_(True)
    wr, br = w.double().requires_grad_(True), be.double().requires_grad_(True)
    want = F.layer_norm(s, (C,), wr, br, norm.eps)
    if add:
        su, n = add_layer_norm(ad, bd, norm)
        assert torch.equal(su.cpu(), a + b)
        torch.autograd.backward([su, n], [ds.to(DEV), dn.to(DEV)])
        torch.autograd.backward([want, s * 1.0], [dn.double(), ds.double()])
    else:
        n = layer_norm(ad, norm)
        n.backward(dn.to(DEV))
        want.backward(dn.double())
    # one rounding of the result (2^-8 / 2^-11 relative), fp32 statistics (C terms of 2^-24)
    eps = {torch.float32: 2e-6, torch.bfloat16: 2 ** -8, torch.float16: 2 ** -11}[dtype]

    def close(got, ref, scale, what):
        err = (got.detach().double().cpu() - ref).abs()
        assert bool((err <= eps * (ref.abs() + scale)).all()), "%s: %.3e" % (what, float(err.max()))

    close(n, want.detach(), 1.0, "norm")
    close(ad.grad, s.grad, 4.0, "d input")
    if add:
        assert torch.equal(ad.grad, bd.grad)
    # sums over the rows: `rows` terms of size 1, each off by up to 8 * 2^-24 (fp32 mean, deviation,
    # product), signs independent: 4 sigma of sqrt(rows) * 8 * 2^-24 is below 2e-6 * sqrt(rows)
    close(norm.weight.grad, wr.grad, 1.0 + rows ** 0.5, "d weight")
    close(norm.bias.grad, br.grad, 1.0 + rows ** 0.5, "d bias")
    # without autograd the same bits
    with torch.no_grad():
        again = add_layer_norm(ad, bd, norm)[1] if add else layer_norm(ad, norm)
    assert torch.equal(again, n.detach())


def test_add_layer_norm_unused_results():
    """Only one of the two results takes part in the loss."""
    norm = torch.nn.LayerNorm(64).to(DEV)
    a, b = (torch.randn(6, 64, device=DEV, requires_grad=True) for _ in range(2))
    su, _ = add_layer_norm(a, b, norm)
    su.sum().backward()
    assert torch.equal(a.grad, torch.ones_like(a)) and norm.weight.grad is None
    a.grad = None
    add_layer_norm(a, b, norm)[1].square().sum().backward()
    ref = a.detach().clone().requires_grad_(True)
    torch.nn.functional.layer_norm(ref + b.detach(), (64,), norm.weight.detach(), norm.bias.detach()).square().sum().backward()
    assert (a.grad - ref.grad).abs().max() < 1e-4
    assert _lib.lib().hsa_last_error() is not None
