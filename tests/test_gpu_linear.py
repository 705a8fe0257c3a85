"""The projection kernels (csrc/hsa_linear.hip) against fp64 at the edges of their tiles, and the routes to them."""
import ctypes

import pytest
import torch
import torch.nn as nn
import torch.nn.functional as F

import sparseattention_amd as sa
from sparseattention_amd import _lib, transformer
from sparseattention_amd.ops.linear import linear, query_key_value

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Segment(ctypes.Structure):
    _fields_ = ([(n, ctypes.c_void_p) for n in ("x", "w", "bias", "out")]
                + [(n, ctypes.c_int64) for n in ("ld_x", "ld_w", "ld_out", "batch_x", "batch_out")]
                + [(n, ctypes.c_int) for n in ("batches", "rows", "cols")])


def _segment(x, w, bias, out):
    return Segment(x.data_ptr(), w.data_ptr(), None if bias is None else bias.data_ptr(), out.data_ptr(), x.stride(1),
                   w.stride(0), out.stride(1), x.stride(0), out.stride(0), x.shape[0], x.shape[1], out.shape[2])


def _call(segs, K, contract, tile, dtype):
    arr = (Segment * len(segs))(*segs)
    rc = _lib.lib().hsa_linear(len(segs), arr, K, int(contract), tile, 1 if dtype == torch.float16 else 2,
                               ctypes.c_void_p(torch.cuda.current_stream().cuda_stream))
    _lib.check(rc, "hsa_linear")


def _bound(x, w, ref, dtype):
    """One rounding of the result (half a unit in the last place, half the smallest subnormal below) and K fp32
    additions and products, each off by at most 2^-24 of the sum of magnitudes."""
    half = 2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8  # 10 and 7 stored bits
    sums = x.double().abs() @ w.double().abs()
    return half * ref.abs() * 1.01 + 2.0 ** -25 + x.shape[-1] * 2.0 ** -23 * (sums + 1)


def _check(dtype, contract, tile, B, R, N, K, pad, first):
    """Two projections of one launch, one with a bias and one without, into the middle of larger buffers."""
    g = torch.Generator(DEV).manual_seed(B + R + N + K)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    x, w, bias = mk(B, R, K), mk(K, N) if contract else mk(N, K), mk(N + 1)[1:]
    ld = N + pad
    bufs = [torch.full((B * (R + 1) * ld + 64,), 7.0, device=DEV, dtype=dtype) for _ in range(2)]
    outs = [b.as_strided((B, R, N), ((R + 1) * ld, ld, 1), first) for b in bufs]
    _call([_segment(x, w, bias, outs[0]), _segment(x, w, None, outs[1])][:1 if tile == 4 else 2], K, contract, tile, dtype)
    wt = w if contract else w.t()
    ref = x.double() @ wt.double()
    for i, want in enumerate((ref + bias.double(), ref)[:1 if tile == 4 else 2]):
        err = (outs[i].double() - want).abs()
        assert bool((err <= _bound(x, wt, want, dtype)).all()), (i, float(err.max()))
        rest = bufs[i].clone()
        rest.as_strided((B, R, N), ((R + 1) * ld, ld, 1), first).fill_(7.0)
        assert bool((rest == 7).all()), "written outside the result"


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("contract", [False, True])
@pytest.mark.parametrize("tile,B,R,N,K", [
    (0, 1, 256, 256, 128), (0, 3, 257, 264, 192), (0, 2, 511, 512, 320), (0, 1, 8448, 520, 128),
    (1, 1, 256, 192, 128), (1, 2, 300, 200, 512), (1, 5, 257, 392, 192),
    (2, 1, 128, 128, 128), (2, 3, 130, 136, 192), (2, 1, 4099, 768, 128)])
def test_tiles_against_fp64(dtype, contract, tile, B, R, N, K):
    _check(dtype, contract, tile, B, R, N, K, 8, 16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,R,N,K", [(1, 1, 4, 32), (2, 17, 36, 64), (1, 33, 32, 96), (3, 31, 100, 672), (1, 256, 512, 2080)])
def test_few_rows_against_fp64(dtype, B, R, N, K):
    _check(dtype, False, 3, B, R, N, K, (8 - N % 8) % 8 + 8, 16)


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("B,R,N,K,pad,first", [
    (1, 256, 256, 128, 0, 0), (2, 257, 257, 192, 0, 3), (1, 300, 511, 512, 2, 1), (1, 512, 1000, 128, 3, 7),
    (1, 16384, 257, 128, 0, 0), (1, 16447, 513, 192, 2, 5), (1, 8300, 320, 128, 2, 1),
    (1, 16384, 8191, 128, 0, 0), (1, 16384, 8192, 128, 1, 5), (1, 16384, 8130, 192, 1, 63), (1, 8192, 8190, 128, 0, 1),
    (1, 8192, 8187, 128, 3, 58), (1, 4096, 8188, 128, 0, 0), (1, 28675, 7938, 128, 2, 31), (1, 16384, 8001, 192, 0, 3)])
def test_results_that_begin_anywhere(dtype, B, R, N, K, pad, first):
    """Rows through the LDS; from 7937 columns and 256 rows per line period on (16384 for odd strides, 8192 for twice an
    odd one, 4096 for four times one) tiles of rows that lie alike, which begin up to 63 columns before their place."""
    _check(dtype, False, 4, B, R, N, K, pad, first)


def test_refused_sizes():
    x, w = torch.zeros(1, 256, 128, device=DEV, dtype=torch.bfloat16), torch.zeros(256, 128, device=DEV, dtype=torch.bfloat16)
    out = torch.empty(1, 256, 256, device=DEV, dtype=torch.bfloat16)
    ok = _segment(x, w, None, out)
    tile = _lib.lib().hsa_linear_tile
    assert tile(1, ctypes.byref(ok), 128, 0, 0) == -1  # fp32
    assert tile(0, ctypes.byref(ok), 128, 0, 2) == -1
    for kind, K, name, value in ((0, 96, None, 0), (0, 128, "rows", 255), (0, 128, "cols", 248), (0, 128, "ld_out", 260),
                                 (0, 128, "ld_x", 120), (3, 33, None, 0), (4, 128, "cols", 255)):
        s = _segment(x, w, None, out)
        if name:
            setattr(s, name, value)
        with pytest.raises(_lib.HsaError):
            _call([s], K, False, kind, torch.bfloat16)
    with pytest.raises(_lib.HsaError):
        _call([ok], 128, True, 3, torch.bfloat16)


@pytest.mark.parametrize("rows,cols,K,bias", [(8192, 1536, 512, False), (256, 512, 512, True), (4096, 10001, 256, True),
                                              (64, 40, 96, True)])
def test_linear_without_autograd(rows, cols, K, bias):
    """Each route, chosen by the sizes: tiles, few rows, results that begin anywhere."""
    torch.manual_seed(0)
    layer = nn.Linear(K, cols, bias=bias).to(DEV, torch.bfloat16)
    x = torch.randn(2, rows // 2, K, device=DEV, dtype=torch.bfloat16)
    with torch.no_grad():
        got = linear(layer, x)
        strided = x.transpose(0, 1).contiguous().transpose(0, 1)  # rows that lie apart: the layer itself
        assert torch.equal(linear(layer, strided), layer(strided))
    wt = layer.weight.detach().t()
    want = x.double() @ wt.double() + (layer.bias.detach().double() if bias else 0)
    assert got.shape == want.shape and got.dtype == torch.bfloat16 and not got.requires_grad
    assert bool(((got.double() - want).abs() <= _bound(x, wt, want, torch.bfloat16)).all())


@pytest.mark.filterwarnings("ignore:Sparse CSR")
def test_weight_without_strides():
    """A weight held as compressed sparse rows has no strides to ask for: the layer's own product."""
    layer = nn.Linear(64, 32, bias=False).to(DEV)
    layer.weight = nn.Parameter(layer.weight.detach().to_sparse_csr(), requires_grad=False)
    x = torch.randn(48, 64, device=DEV)
    with torch.no_grad():
        got = linear(layer, x)
    want = x.double() @ layer.weight.to_dense().double().t()
    # K products and additions in fp32
    assert bool(((got.double() - want).abs() <= 64 * 2.0 ** -23 * (x.double().abs() @ layer.weight.to_dense().double().abs().t())).all())


@pytest.mark.parametrize("rows,K,cols", [(16384, 512, 512), (64, 96, 40)])
@pytest.mark.parametrize("contract", [False, True])
def test_products_with_a_bias(rows, K, cols, contract):
    """Kernel and library, chosen by the sizes: the same sum on either route."""
    torch.manual_seed(0)
    mk = lambda *s: torch.randn(*s, device=DEV, dtype=torch.bfloat16)
    x, w, b = mk(rows, K), mk(K, cols) if contract else mk(cols, K), mk(cols)
    wt = w if contract else w.t()
    got, want = _lib.ext().project(x, w, b, contract), x.double() @ wt.double() + b.double()
    assert bool(((got.double() - want).abs() <= _bound(x, wt, want, torch.bfloat16)).all())


@pytest.mark.parametrize("amp", [None, torch.float16])
@pytest.mark.parametrize("B,N,C", [(1, 64, 64), (2, 256, 256), (4, 1024, 512)])
def test_query_key_value(amp, B, N, C):
    torch.manual_seed(0)
    dtype = torch.float32 if amp else torch.bfloat16
    layers = [nn.Linear(C, C, bias=False).to(DEV, dtype) for _ in range(3)]
    x, y = torch.randn(B, N, C, device=DEV).to(dtype), torch.randn(B, N - 1, C, device=DEV).to(dtype)
    with torch.no_grad(), torch.autocast("cuda", dtype=amp or torch.float16, enabled=amp is not None):
        got = query_key_value(*layers, x, y)
    low = amp or dtype
    assert got is not None
    for i, (t, layer) in enumerate(zip(got, layers)):
        rows = (x if i == 0 else torch.cat([x, y], dim=1)).to(low)
        wt = layer.weight.detach().to(low).t()
        want = rows.double() @ wt.double()
        assert t.dtype == low and t.is_contiguous() and t.shape == want.shape
        assert bool(((t.double() - want).abs() <= _bound(rows, wt, want, low)).all())
    x.requires_grad_(True)
    assert query_key_value(*layers, x, y) is None  # not with autograd


def test_input_gradient_on_tiles():
    """The input gradient of a projection that is large enough for the kernel, against fp64."""
    torch.manual_seed(0)
    layer = nn.Linear(512, 512).to(DEV, torch.bfloat16)
    x = torch.randn(16384, 512, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    dy = torch.randn(16384, 512, device=DEV, dtype=torch.bfloat16)
    linear(layer, x).backward(dy)
    w = layer.weight.detach()
    want = dy.double() @ w.double()
    assert bool(((x.grad.double() - want).abs() <= _bound(dy, w, want, torch.bfloat16)).all())


def test_replays_of_a_graph_with_projections():
    torch.manual_seed(0)
    layer = nn.Linear(256, 1024).to(DEV, torch.bfloat16)
    small, large = (torch.randn(n, 256, device=DEV, dtype=torch.bfloat16) for n in (64, 8192))
    with torch.no_grad():
        s = torch.cuda.Stream()
        with torch.cuda.stream(s):
            linear(layer, small), linear(layer, large)
        torch.cuda.current_stream().wait_stream(s)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            outs = linear(layer, small), linear(layer, large)
        for i in range(3):
            small.normal_(), large.normal_()
            graph.replay()
            torch.cuda.synchronize()
            assert torch.equal(outs[0], linear(layer, small)) and torch.equal(outs[1], linear(layer, large))


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("M,N,K", [(256, 256, 128), (257, 264, 129), (300, 512, 1001), (511, 1000, 777), (256, 256, 16385)])
def test_long_contraction_against_fp64(dtype, M, N, K):
    """Parts of the contraction that end within a step, rows that begin at any element, tiles flush with the end.
    What lies behind a row's end and behind the weight's last row is not read as a number."""
    g = torch.Generator(DEV).manual_seed(K)
    mk = lambda *s: torch.randn(*s, generator=g, device=DEV).to(dtype)
    x, w = mk(M, K + 5), mk(K + 64, N)
    x[:, 0], x[:, K + 1:] = float("nan"), float("nan")
    w[K:] = float("inf")
    x, w = x[:, 1:K + 1], w[:K]
    lib, code = _lib.lib(), 1 if dtype == torch.float16 else 2
    ws = torch.empty(lib.hsa_linear_long_workspace_bytes(M, N, K, code) // 4, device=DEV)
    out = torch.empty(M, N + 8, device=DEV, dtype=dtype)[:, :N]
    args = (x.data_ptr(), K + 5, w.data_ptr(), N, out.data_ptr(), N + 8, M, N, K, ws.data_ptr())
    stream = ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)
    _lib.check(lib.hsa_linear_long(*args, ws.numel() * 4, code, stream), "hsa_linear_long")
    ref = x.double() @ w.double()
    assert bool(((out.double() - ref).abs() <= _bound(x, w, ref, dtype)).all())
    with pytest.raises(_lib.HsaError):
        _lib.check(lib.hsa_linear_long(*args, ws.numel() * 4 - 4, code, stream), "hsa_linear_long")


def test_model_with_a_vocabulary_whose_last_tile_is_nearly_full(monkeypatch):
    """50428 columns (252 in the last tile of 256) of 4 x 1024 rows: logits and loss, with and without autograd, against
    the layer's own product; the results' memory held NaN before."""
    vocab, B, N = 50428, 4, 1024
    torch.manual_seed(0)
    net = sa.TransformerLM(vocab, 128, 2, 128, 1, dropout=0.0, window_size=4, max_len=N).to(DEV).to(torch.bfloat16)
    tok, to = (torch.randint(0, vocab, (B, N), device=DEV) for _ in range(2))

    def run():
        torch.full((B * N * vocab,), float("nan"), device=DEV, dtype=torch.bfloat16)
        logits = net(tok)
        return logits, F.cross_entropy(logits.float().view(-1, vocab), to.view(-1))

    def both():
        net.zero_grad(set_to_none=True)
        with torch.no_grad():
            plain = run()
        logits, loss = run()
        loss.backward()
        return plain + (logits.detach(), loss.detach()), [p.grad.float() for p in net.parameters() if p.grad is not None]

    got, grads = both()
    with monkeypatch.context() as m:
        m.setattr(transformer, "linear", lambda layer, x, wide=False: layer(x))
        want, want_grads = both()
    for a, b in zip(got, want):  # one rounding to bf16 on either side of sums of 128 products
        assert bool(((a.float() - b.float()).abs() <= 2.0 ** -7 * b.float().abs() + 1e-4).all())
    for a, b in zip(grads, want_grads):  # the logits' roundings carried back through a softmax: a hundredth
        assert float((a - b).norm()) <= 0.01 * float(b.norm()) + 1e-12


@pytest.mark.parametrize("vocab", [50257, 5120])
def test_vocabulary_projection_in_training(vocab):
    """Forward and all three gradients against fp64, and a second derivative against the layer's own."""
    torch.manual_seed(0)
    layer = nn.Linear(256, vocab).to(DEV, torch.bfloat16)
    x = torch.randn(2, 512, 256, device=DEV, dtype=torch.bfloat16, requires_grad=True)
    y = linear(layer, x, wide=True)
    w, b = layer.weight.detach(), layer.bias.detach()
    assert bool(((y.double() - (x.double() @ w.double().t() + b.double())).abs() <= _bound(x.detach(), w.t(), y.detach().double(), torch.bfloat16)).all())
    dy = torch.randn_like(y)
    y.backward(dy)
    g, r = dy.reshape(-1, vocab), x.detach().reshape(-1, 256)
    want = g.double() @ w.double()
    assert bool(((x.grad.reshape(-1, 256).double() - want).abs() <= _bound(g, w, want, torch.bfloat16)).all())
    want = g.double().t() @ r.double()
    assert bool(((layer.weight.grad.double() - want).abs() <= _bound(g.t(), r, want, torch.bfloat16)).all())
    want = g.double().sum(0)
    assert bool(((layer.bias.grad.double() - want).abs() <= 2.0 ** -8 * 1.01 * want.abs() + 1024 * 2.0 ** -23 * g.double().abs().sum(0)).all())
    second = []
    for f in (lambda: linear(layer, x, wide=True), lambda: layer(x)):
        x.grad = None
        d, = torch.autograd.grad(f().float().square().mean(), x, create_graph=True)
        d.float().square().mean().backward()
        second.append(x.grad.float())
    # bf16 on both sides, two products deep: a hundredth of the norm
    assert float((second[0] - second[1]).norm()) <= 0.01 * float(second[1].norm()) and float(second[1].norm()) > 0
