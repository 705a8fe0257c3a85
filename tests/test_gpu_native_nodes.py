"""The native calls keep what the calls they stand in for did: second derivatives, replaced and watched modules,
in-place updates, batched gradients, refusals."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import _lib
from sparseattention_amd.ops import functional as fn
from sparseattention_amd.ops.linear import linear, query_key_value, query_key_value_rows
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


@pytest.mark.parametrize("one_pass", [None, False])
def test_attention_differentiated_twice_says_so(one_pass):
    """The span attention has no second derivative: its first one is there with create_graph, and what needs the
    second raises instead of leaving its terms out."""
    B, N, H, D = 1, 64, 2, 32
    t = sa.build_tree_topology(N, True, device=DEV)
    q, k, v = (torch.randn(B, n, H, D, device=DEV, dtype=torch.bfloat16, requires_grad=True) for n in (N, 2 * N - 1, 2 * N - 1))
    w = torch.randn(D, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    old, fn.one_pass_backward = fn.one_pass_backward, one_pass
    try:
        run = lambda: (sa.hierarchical_attention(q, k, v, t["forward_idx"], t["backward_gather"], t["forward_mask"], 4) * w).sum()
        want = torch.autograd.grad(run(), [q, k, v, w])
        got = torch.autograd.grad(run(), [q, k, v, w], create_graph=True)
        assert all(torch.equal(a, b) for a, b in zip(want, got))
        # the part of the graph in front of the attention is differentiated as before
        assert torch.equal(torch.autograd.grad(got[3].sum(), q, retain_graph=True)[0].isfinite().all(), torch.tensor(True, device=DEV))
        with pytest.raises(RuntimeError, match="differentiat"):
            torch.autograd.grad(got[0].float().sum(), [k])
    finally:
        fn.one_pass_backward = old


# ------------------------------------------------------------------------- replaced and watched modules
def _small_lm():
    torch.manual_seed(0)
    return sa.TransformerLM(50, 64, 2, 128, 2, dropout=0.0, window_size=4, max_len=32).to(DEV).to(torch.bfloat16)


def test_a_replaced_forward_runs():
    """A forward set on the instance (what checkpointing and offloading helpers do) is called, of layers and norms."""
    net = _small_lm()
    tok = torch.randint(0, 50, (1, 32), device=DEV)
    want = net(tok)
    for module in (net.layers[1], net.layers[0].norm1, net.layers[1].norm2, net.layers[1].norm_y, net.layers[1].feed_forward.fc1):
        seen, inner = [], module.forward

        def forward(*args, **kwargs):
            seen.append(1)
            return inner(*args, **kwargs)

        module.forward = forward
        got = net(tok)
        del module.forward
        assert seen, type(module)
        # the layer's own code path in place of the chained one: single roundings
        assert (got.float() - want.float()).norm() <= 2e-2 * want.float().norm()
    assert torch.equal(net(tok), want)


@pytest.mark.parametrize("register", [torch.nn.modules.module.register_module_forward_hook,
                                      torch.nn.modules.module.register_module_forward_pre_hook,
                                      torch.nn.modules.module.register_module_full_backward_hook])
def test_global_module_hooks_see_every_module(register):
    net = _small_lm()
    tok = torch.randint(0, 50, (1, 32), device=DEV)
    seen = []
    handle = register(lambda m, *args: seen.append(m))
    try:
        net(tok).float().sum().backward()
    finally:
        handle.remove()
    for layer in net.layers:
        for m in (layer, layer.norm1, layer.norm2, layer.norm_y, layer.feed_forward.fc1):
            assert any(m is s for s in seen), type(m)


# ------------------------------------------------------------------------- what a backward needs
@pytest.mark.parametrize("amp", [torch.float16, torch.bfloat16])
def test_autocast_backward_after_an_update(amp):
    """Under autocast the backward works from 16-bit copies: the fp32 parameters and activations may be written
    to in between (an in-place residual sum, an optimizer step between two backwards)."""
    lq, lk, lv = (torch.nn.Linear(64, 64, bias=False).to(DEV) for _ in range(3))
    lin = torch.nn.Linear(64, 96).to(DEV)
    x0, y0 = torch.randn(2, 8, 64, device=DEV), torch.randn(2, 7, 64, device=DEV)
    params = [lq.weight, lk.weight, lv.weight, lin.weight, lin.bias]

    def run(update):
        leaves = [x0.clone().requires_grad_(True), y0.clone().requires_grad_(True)]
        x, y = leaves[0] * 1.0, leaves[1] * 1.0
        with torch.autocast("cuda", dtype=amp):
            q, k, v = query_key_value_rows(lq, lk, lv, x, y)
            z = linear(lin, x)
        loss = sum((t.float() ** 2).sum() for t in (q, k, v, z))
        if update:
            with torch.no_grad():
                x.add_(1.0)
                y.add_(1.0)
                for p in params:
                    p.add_(1.0)
        grads = torch.autograd.grad(loss, leaves + params)
        if update:
            with torch.no_grad():
                for p in params:
                    p.sub_(1.0)
        return grads

    want = run(False)
    kept = [p.detach().clone() for p in params]
    got = run(True)
    with torch.no_grad():
        for p, old in zip(params, kept):
            p.copy_(old)
    assert all(torch.equal(a, b) for a, b in zip(want, got))


def test_autocast_keeps_no_fp32_activations():
    """The rows' fp32 originals are free once their 16-bit copies are made."""
    lq, lk, lv = (torch.nn.Linear(64, 64, bias=False).to(DEV) for _ in range(3))
    leaf = torch.randn(4, 4096, 64, device=DEV, requires_grad=True)
    y = torch.randn(4, 4095, 64, device=DEV, dtype=torch.float16)
    x = leaf * 1.0
    bytes_x = x.numel() * 4
    with torch.autocast("cuda", dtype=torch.float16):
        out = query_key_value_rows(lq, lk, lv, x, y)
    before = torch.cuda.memory_allocated()
    del x
    assert before - torch.cuda.memory_allocated() >= bytes_x
    sum(t.float().sum() for t in out).backward()
    assert leaf.grad is not None


def test_autocast_backward_differentiated_twice():
    """The saved 16-bit copies lead back to the fp32 activations and parameters."""
    lq, lk, lv, lin = (torch.nn.Linear(64, 64, bias=False).to(DEV) for _ in range(4))
    x, y = (torch.randn(2, n, 64, device=DEV, requires_grad=True) for n in (8, 7))

    def second(f):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            q, k, v, z = f()
        first = torch.autograd.grad(sum((t.float() ** 3).sum() for t in (q, k, v, z)), [x, y, lk.weight], create_graph=True)
        leaves = [x, y, lq.weight, lk.weight, lv.weight, lin.weight]
        return torch.autograd.grad(sum((g ** 2).sum() for g in first), leaves, allow_unused=True)

    def plain():
        xy = torch.cat([x, y], dim=1)
        return lq(x), lk(xy), lv(xy), lin(x)

    for a, b in zip(second(lambda: (*query_key_value_rows(lq, lk, lv, x, y), linear(lin, x))), second(plain)):
        # bf16 through two backward passes, summed in other orders: a few units of 2^-8 of the norm
        assert a.dtype == b.dtype and (a - b).norm() <= 2e-2 * b.norm()


# ------------------------------------------------------------------------- batched gradients, wrapped parameters
def test_batched_gradients():
    """vmap over the gradients of the outputs (is_grads_batched) through the norm and the linear layers."""
    B, C, n = 2, 64, 3
    lq, lk, lv = (torch.nn.Linear(C, C, bias=False).to(DEV).to(torch.bfloat16) for _ in range(3))
    lin, norm = (m.to(DEV).to(torch.bfloat16) for m in (torch.nn.Linear(C, 96), torch.nn.LayerNorm(C)))
    mk = lambda *s: torch.randn(*s, device=DEV, dtype=torch.bfloat16)
    x, y, b = (mk(B, m, C).requires_grad_(True) for m in (8, 7, 8))
    calls = {"linear": (lambda: [linear(lin, x)], [x, lin.weight, lin.bias]),
             "norm": (lambda: [layer_norm(x, norm)], [x, norm.weight, norm.bias]),
             "sum and norm": (lambda: list(add_layer_norm(x, b, norm)), [x, b, norm.weight, norm.bias]),
             "rows": (lambda: list(query_key_value_rows(lq, lk, lv, x, y)), [x, y, lq.weight, lk.weight, lv.weight])}
    for name, (call, leaves) in calls.items():
        outs = call()
        gs = [mk(n, *o.shape) for o in outs]
        got = torch.autograd.grad(outs, leaves, gs, is_grads_batched=True, retain_graph=True)
        for i in range(n):
            for a, w in zip(got, torch.autograd.grad(call(), leaves, [g[i] for g in gs])):
                # bf16: a few roundings of 2^-9 more or less
                assert (a[i].float() - w.float()).norm() <= 2e-2 * w.float().norm(), name


class _Normed(torch.nn.Module):
    def __init__(self):
        super().__init__()
        self.norm = torch.nn.LayerNorm(64)

    def forward(self, x, b):
        return add_layer_norm(x, b, self.norm)[1] + layer_norm(x, self.norm)


def test_norm_with_wrapped_parameters():
    """A functional transform over the norm's parameters (an ensemble of weights) goes through torch's own norm."""
    net = _Normed().to(DEV)
    x, b = torch.randn(5, 64, device=DEV), torch.randn(5, 64, device=DEV)
    ws, bs = torch.randn(3, 64, device=DEV), torch.randn(3, 64, device=DEV)
    one = lambda w, c: torch.func.functional_call(net, {"norm.weight": w, "norm.bias": c}, (x, b))
    got = torch.func.vmap(one)(ws, bs)
    for i in range(3):
        assert (got[i] - one(ws[i], bs[i])).abs().max() < 1e-4
    g = torch.func.grad(lambda w: one(w, bs[0]).square().sum())(ws[0])
    w = ws[0].clone().requires_grad_(True)
    assert (g - torch.autograd.grad(one(w, bs[0]).square().sum(), w)[0]).abs().max() < 1e-3


# ------------------------------------------------------------------------- refusals
@pytest.mark.parametrize("dtype,grad", [(torch.bfloat16, False), (torch.float32, False), (torch.float32, True)])
def test_tables_on_the_host_are_refused(dtype, grad):
    """(The one-pass training forward takes them: it never looked at the tables' place.)"""
    B, N, H, D = 1, 64, 2, 32
    q, k, v = (torch.randn(B, n, H, D, device=DEV, dtype=dtype, requires_grad=grad) for n in (N, 2 * N - 1, 2 * N - 1))
    gpu, cpu = sa.build_tree_topology(N, True, device=DEV), sa.build_tree_topology(N, True, device="cpu")
    for idx, mask in ((cpu, cpu), (cpu, gpu), (gpu, cpu)):
        with pytest.raises(_lib.HsaError):
            sa.hierarchical_attention(q, k, v, idx["forward_idx"], gpu["backward_gather"], mask["forward_mask"], 4)
    with pytest.raises(_lib.HsaError):
        sa.hierarchical_attention(q, k, v, cpu["forward_idx"], gpu["backward_gather"], None, 4)


def test_errors_of_the_library_keep_their_type():
    """What the library itself refuses is an HsaError on the native route too."""
    B, N, H, D = 1, 64, 1, 32
    t = sa.build_tree_topology(N, True, device=DEV)
    q, k, v = (torch.randn(B, n, H, D, device=DEV, dtype=torch.bfloat16) for n in (N, 2 * N - 1, 2 * N - 1))
    for grad in (False, True):
        q.requires_grad_(grad)
        with pytest.raises(_lib.HsaError, match="slots"):  # 2R+1+L beyond the gather kernel's 256 slots
            sa.hierarchical_attention(q, k, v, t["forward_idx"], t["backward_gather"], t["forward_mask"], 200)
    with pytest.raises(AssertionError):
        sa.hierarchical_attention(q.detach()[0, :, 0, 0], k, v, t["forward_idx"], t["backward_gather"], t["forward_mask"], 4)


# ------------------------------------------------------------------------- watched calls
class _Seen(torch.overrides.TorchFunctionMode):
    """Counts the functions called under it."""

    def __init__(self):
        super().__init__()
        self.calls = []

    def __torch_function__(self, func, types, args=(), kwargs=None):
        self.calls.append(func)
        return func(*args, **(kwargs or {}))


class _Tagged(torch.Tensor):
    pass


def _small_model():
    torch.manual_seed(0)
    return sa.TransformerLM(50, 128, 2, 128, 2, dropout=0.0, window_size=4, max_len=64).to(DEV).to(torch.bfloat16).eval()


@pytest.mark.parametrize("train", [False, True])
def test_function_modes_see_the_calls(train):
    """A mode that handles torch's functions is given the projections and norms, with and without autograd; a default
    device, which is such a mode too, changes nothing."""
    net, tok = _small_model(), torch.randint(0, 50, (2, 64), device=DEV)
    with torch.set_grad_enabled(train):
        want = net(tok)
        with _Seen() as seen:
            got = net(tok)
        # the last projection and, a layer, seven products besides those that the span nodes share
        assert seen.calls.count(torch.nn.functional.linear) >= 15
        assert seen.calls.count(torch.nn.functional.layer_norm) == 6
        assert (got.float() - want.float()).norm() <= 0.03 * want.float().norm()
        with torch.device(DEV):
            assert torch.equal(net(tok), want)


def test_subclasses_that_handle_functions_are_kept():
    """The layer's own call gives back the subclass; so does the native route in its place."""
    layer, norm = torch.nn.Linear(128, 64).to(DEV, torch.bfloat16), torch.nn.LayerNorm(128).to(DEV, torch.bfloat16)
    x = torch.randn(2, 32, 128, device=DEV, dtype=torch.bfloat16)
    t = x.as_subclass(_Tagged)
    for grad in (False, True):
        with torch.set_grad_enabled(grad):
            assert type(linear(layer, t)) is _Tagged and type(layer_norm(t, norm)) is _Tagged
            assert type(linear(layer, x)) is torch.Tensor
    with torch.no_grad():
        layers = [torch.nn.Linear(128, 128, bias=False).to(DEV, torch.bfloat16) for _ in range(3)]
        assert query_key_value(*layers, t, t) is None and query_key_value(*layers, x, x) is not None


def test_dispatch_modes_see_the_products():
    """The products inside the span nodes' update count for a mode that watches dispatched calls."""
    from torch.utils.flop_counter import FlopCounterMode
    net, B, N, C = _small_model(), 2, 64, 128
    x, y = torch.randn(B, N, C, device=DEV, dtype=torch.bfloat16), torch.randn(B, N - 1, C, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad(), FlopCounterMode(display=False) as counter:
        net.layers[0].self_attn.cross_update_Y(x, y)
    assert counter.get_total_flops() >= 2 * B * (N - 1) * C * 4 * C  # q, k, v of the nodes and the last projection
