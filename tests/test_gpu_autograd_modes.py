"""The native calls under autograd's less common modes: forward-mode tangents, hooks on saved tensors."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd.ops.linear import linear
from sparseattention_amd.transformer import layer_norm

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def test_native_calls_refuse_tangents():
    """A forward-mode tangent is not dropped: the span attention has no rule for it and says so."""
    B, N, H, D = 1, 16, 2, 32
    t = sa.build_tree_topology(N, True, device=DEV)
    q, k, v = torch.randn(B, N, H, D, device=DEV), *(torch.randn(B, 2 * N - 1, H, D, device=DEV) for _ in range(2))
    with torch.autograd.forward_ad.dual_level():
        d = torch.autograd.forward_ad.make_dual(q, torch.ones_like(q))
        with pytest.raises(RuntimeError):
            sa.hierarchical_attention(d, k, v, t["forward_idx"], t["backward_gather"], t["forward_mask"], 4)
        norm = torch.nn.LayerNorm(D).to(DEV)
        assert torch.autograd.forward_ad.unpack_dual(layer_norm(d, norm)).tangent is not None


def test_saved_tensors_with_another_layout():
    """Hooks that give saved tensors back with other strides change nothing."""
    B, N, H, D = 2, 64, 2, 32
    t = sa.build_tree_topology(N, True, device=DEV)
    mk = lambda n: torch.randn(B, n, H, D, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    q, k, v = mk(N), mk(2 * N - 1), mk(2 * N - 1)
    norm = torch.nn.LayerNorm(D).to(DEV).to(torch.bfloat16)
    lin = torch.nn.Linear(D, D).to(DEV).to(torch.bfloat16)

    def grads():
        o = sa.hierarchical_attention(q, k, v, t["forward_idx"], t["backward_gather"], t["forward_mask"], 4)
        return torch.autograd.grad(linear(lin, layer_norm(o, norm)).float().square().sum(), [q, k, v, lin.weight, lin.bias])

    want = grads()
    turn = lambda s: s.transpose(0, -1).contiguous().transpose(0, -1)
    with torch.autograd.graph.saved_tensors_hooks(turn, lambda s: s):
        got = grads()
    for a, b in zip(got, want):
        assert torch.equal(a, b)


def test_span_levels_saved_with_another_layout():
    """The same for the span-node update, chains of small levels included."""
    net = sa.HierarchicalAttention(128, 2, dropout=0.0).to(DEV).to(torch.bfloat16)
    net._TRAINING_CHAIN_ROWS = 64
    x, y = (torch.randn(2, n, 128, device=DEV, dtype=torch.bfloat16, requires_grad=True) for n in (128, 127))

    def grads():
        return torch.autograd.grad(net.cross_update_Y(x, y).float().square().sum(), [x, y, net.Wk_y.weight, net.Wq_y.weight])

    want = grads()
    turn = lambda s: s.transpose(0, -1).contiguous().transpose(0, -1)
    with torch.autograd.graph.saved_tensors_hooks(turn, lambda s: s):
        got = grads()
    for a, b in zip(got, want):
        assert torch.equal(a, b)
