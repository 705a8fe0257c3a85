"""The decoder layer as one native call (csrc/torch_ops.cpp) against the Python layer it stands in for, and the cases
in which it does not."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import transformer
from sparseattention_amd.modules import attention

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _lm(dim=128, heads=2, ff=128, layers=2, act="gelu", dtype=torch.bfloat16, length=64, dropout=0.0):
    torch.manual_seed(0)
    return sa.TransformerLM(50, dim, heads, ff, layers, dropout=dropout, window_size=4, activation=act,
                            max_len=length).to(DEV).to(dtype).eval()


class _Count:
    """How many layers ran natively."""

    def __init__(self, monkeypatch):
        self.native = 0
        inner = transformer.DecoderLayer._native

        def counted(layer, *args, **kwargs):
            r = inner(layer, *args, **kwargs)
            self.native += r is not None
            return r

        monkeypatch.setattr(transformer.DecoderLayer, "_native", counted)


def _python(net, tok, monkeypatch):
    with monkeypatch.context() as m:
        m.setattr(transformer.DecoderLayer, "_native", lambda self, *a, **k: None)
        return net(tok)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("act", ["gelu", "relu"])
@pytest.mark.parametrize("B,N,dim,heads,ff", [(1, 2, 128, 4, 128), (1, 64, 64, 2, 128), (3, 256, 512, 8, 2048), (2, 128, 384, 3, 1000),
                                              (8, 1024, 256, 4, 512), (1, 512, 768, 12, 3072)])
def test_same_bits_as_the_python_layer(B, N, dim, heads, ff, act, dtype, monkeypatch):
    net, tok = _lm(dim, heads, ff, 3, act, dtype, N), torch.randint(0, 50, (B, N), device=DEV)
    count = _Count(monkeypatch)
    with torch.no_grad():
        got = net(tok)
        handled = sa._lib.lib().hsa_cross_update_level_rows(B, heads, dim // heads, 2) >= N
        assert count.native == (3 if handled else 0)
        assert torch.equal(got, _python(net, tok, monkeypatch))
        # other weights
        for p in net.parameters():
            p.mul_(0.5)
        assert torch.equal(net(tok), _python(net, tok, monkeypatch))


def test_calls_that_stay_with_the_python_layer(monkeypatch):
    net, tok = _lm(), torch.randint(0, 50, (2, 64), device=DEV)
    count = _Count(monkeypatch)
    with torch.no_grad():
        want = net(tok)
        assert count.native == 2

        def stays(layers, what):
            count.native = 0
            out = net(tok)
            assert count.native == 2 - layers, what
            return out

        layer = net.layers[1]
        for module in (layer.self_attn, layer.feed_forward, layer.norm2, layer.norm_y, layer.self_attn.out_proj_x,
                       layer.self_attn.Wq_x, layer.feed_forward.fc2, layer.feed_forward.dropout):
            seen = []
            handle = module.register_forward_hook(lambda m, *a: seen.append(m))
            # (the second layer's norm_y is taken by the first)
            assert torch.equal(stays(1, type(module)), want) and seen
            handle.remove()
            inner = module.forward
            module.forward = lambda *a, **k: (seen.append(1), inner(*a, **k))[1]
            seen.clear()
            assert torch.equal(stays(1, type(module)), want) and seen
            del module.forward
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: None)
        stays(2, "global hook")
        handle.remove()
        calls = []
        with monkeypatch.context() as m:
            inner = attention.HierarchicalAttention.cross_update_Y
            m.setattr(attention.HierarchicalAttention, "cross_update_Y", lambda *a, **k: (calls.append(1), inner(*a, **k))[1])
            assert torch.equal(stays(2, "class"), want) and len(calls) == 2
        with monkeypatch.context() as m:
            op = attention.hierarchical_attention
            m.setattr(attention, "hierarchical_attention", lambda *a, **k: (calls.append(1), op(*a, **k))[1])
            assert torch.equal(stays(2, "op"), want) and len(calls) == 4
        layer.self_attn.fuse_top_levels = False
        stays(1, "levels by themselves")
        layer.self_attn.fuse_top_levels = True
        layer.feed_forward.activation = lambda t: t * 2
        assert not torch.equal(stays(1, "activation"), want)
        layer.feed_forward.activation = torch.nn.functional.gelu
        with torch.autocast("cuda", dtype=torch.float16):
            stays(2, "autocast")
        params = {k: v.detach() * 0.5 for k, v in net.named_parameters()}
        count.native = 0
        halved = torch.func.functional_call(net, params, (tok,))
        assert count.native == 0 and not torch.equal(halved, want)
        assert torch.equal(stays(0, "as before"), want)
    count.native = 0
    assert net(tok).requires_grad and count.native == 0


@pytest.mark.parametrize("owner,name,calls", [
    (transformer.PositionwiseFeedForward, "forward", 2), (transformer.DecoderLayer, "_chained", 2), (transformer.DecoderLayer, "forward", 2),
    (attention.HierarchicalAttention, "forward", 2), (attention.HierarchicalAttention, "update_X_from_Y", 2), (torch.nn.LayerNorm, "forward", 6),
    (torch.nn.Linear, "forward", 15), (torch.nn.Dropout, "forward", 11), (transformer, "add_layer_norm", 4), (transformer, "linear", 5),
    (attention, "linear", 4), (attention, "query_key_value", 2)])
def test_steps_replaced_on_their_class_or_module(owner, name, calls, monkeypatch):
    """What stands in a step's place is called, without autograd as in training.  (The results may come from the library's
    products and torch's norms then: bf16 roundings through two layers.)"""
    net, tok = _lm(), torch.randint(0, 50, (2, 64), device=DEV)
    count = _Count(monkeypatch)
    seen, inner = [], getattr(owner, name)
    with torch.no_grad():
        want = net(tok)
        assert count.native == 2
        with monkeypatch.context() as m:
            m.setattr(owner, name, lambda *a, **k: (seen.append(1), inner(*a, **k))[1])
            got = net(tok)
        assert count.native == 2 and len(seen) == calls
        assert float((got.float() - want.float()).norm()) <= 0.03 * float(want.float().norm())
        net(tok)
        assert count.native == 4


@pytest.mark.parametrize("name", ["self_attn.Wq_y", "self_attn.Wk_x", "self_attn.out_proj_y", "feed_forward.fc1", "norm2", "norm1"])
def test_plain_tensors_in_the_parameters_places(name, monkeypatch):
    """Sharding and pruning take a parameter out of its dictionary and keep a plain tensor under its name: the Python
    layer reads that, without autograd (to the same bits) and with it (other products: bf16 roundings through two layers)."""
    net, tok = _lm(), torch.randint(0, 50, (2, 64), device=DEV)
    with torch.no_grad():
        want = net(tok)
    for layer in net.layers:
        m = layer.get_submodule(name)
        for n in list(m._parameters):
            p = m._parameters.pop(n)
            m.__dict__[n] = p if p is None else p.detach().clone()
    count = _Count(monkeypatch)
    with torch.no_grad():
        # (the first layer's own norm1 is not the native layer's, the second's is taken with the first's sums)
        assert torch.equal(net(tok), want) and count.native == (1 if name == "norm1" else 0)
    got = net(tok)
    assert got.requires_grad and float((got.detach() - want).float().norm()) <= 0.03 * float(want.float().norm())


@pytest.mark.parametrize("dim,heads,length", [(768, 12, 1024), (512, 4, 1024), (96, 3, 64)])
def test_sizes_not_taken_are_not_looked_into(dim, heads, length, monkeypatch):
    """What is known from the sizes alone costs no look at the layer's modules."""
    net, tok = _lm(dim, heads, 128, 2, length=length), torch.randint(0, 50, (2, length), device=DEV)
    looks, inner = [], transformer.all_plain
    monkeypatch.setattr(transformer, "all_plain", lambda m: (looks.append(1), inner(m))[1])
    count = _Count(monkeypatch)
    with torch.no_grad():
        net(tok)
    assert count.native == 0 and not looks


def test_dropout_goes_the_python_way(monkeypatch):
    net, tok = _lm(dropout=0.5), torch.randint(0, 50, (2, 64), device=DEV)
    count = _Count(monkeypatch)
    with torch.no_grad():
        a = net(tok)
        assert count.native == 2 and torch.equal(a, net(tok))
        net.train()
        count.native = 0
        assert not torch.equal(net(tok), net(tok)) and count.native == 0


def test_replays_of_a_graph():
    net, tok = _lm(512, 8, 1024, 2, length=256), torch.randint(0, 50, (2, 256), device=DEV)
    with torch.no_grad():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            net(tok)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            out = net(tok)
        for _ in range(3):
            tok.random_(0, 50)
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(out, net(tok))
