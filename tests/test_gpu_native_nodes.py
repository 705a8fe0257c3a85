"""The native calls keep what the calls they stand in for did: second derivatives, replaced and watched modules,
in-place updates, batched gradients, refusals."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import _lib
from sparseattention_amd.ops import functional as fn
from sparseattention_amd.ops.linear import linear, query_key_value_rows
from sparseattention_amd.transformer import add_layer_norm, layer_norm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


# ------------------------------------------------------------------------- differentiated twice
@pytest.mark.parametrize("add", [True, False])
@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_layer_norm_differentiated_twice(add, dtype):
    """A backward that is itself differentiated has the norm's terms, as with torch's own layer norm."""
    norm = torch.nn.LayerNorm(64).to(DEV).to(dtype)
    with torch.no_grad():
        norm.weight.normal_()
        norm.bias.normal_()
    mk = lambda: torch.randn(3, 20, 64, device=DEV, dtype=dtype, requires_grad=True)
    a, b, c = mk(), mk(), mk()
    leaves = [a, norm.weight, norm.bias] + ([b] if add else [])

    def second(f):
        s, n = f()
        first = torch.autograd.grad((n * c).sum() + (n * n).sum() + (s * s * c).sum(), leaves, create_graph=True)
        return torch.autograd.grad(sum((g.float() ** 2).sum() for g in first), leaves + [c])

    def plain():
        s = a + b if add else a
        return s, norm(s)

    def ours():
        return add_layer_norm(a, b, norm) if add else (a, layer_norm(a, norm))

    for x, y in zip(second(ours), second(plain)):
        # bf16: two backward passes of single roundings, in other orders: a few units of 2^-8 of the norm
        assert (x.float() - y.float()).norm() <= (1e-5 if dtype == torch.float32 else 3e-2) * y.float().norm()
