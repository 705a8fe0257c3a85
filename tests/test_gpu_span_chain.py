"""Training: the span-node update's last levels as fused chains, forward and backward."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _run(net, x, y, gy, rows, dtype):
    net._TRAINING_CHAIN_ROWS = rows
    net._fused.clear()
    xl, yl = x.to(dtype).requires_grad_(True), y.to(dtype).requires_grad_(True)
    out = net.cross_update_Y(xl, yl)
    grads = torch.autograd.grad(out, [xl, yl] + [net.Wq_y.weight, net.Wk_y.weight, net.Wv_y.weight], gy.to(dtype))
    return [out.detach()] + list(grads)


# (B, N, heads, head size): chains of one level, from the leaves on, from an inner level on; rows of a tile
# partly filled; contraction lengths that are no multiple of four steps per wavefront; no chain at all
@pytest.mark.parametrize("case", [(1, 2, 2, 64), (3, 16, 8, 32), (2, 64, 4, 64), (5, 256, 6, 64), (1, 512, 4, 128), (3, 1024, 12, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_training_chain(case, dtype):
    B, N, H, Dh = case
    torch.manual_seed(N)
    D = H * Dh
    ref = sa.HierarchicalAttention(D, H, dropout=0.0).to(DEV)
    net = sa.HierarchicalAttention(D, H, dropout=0.0).to(DEV).to(dtype)
    net.load_state_dict({k: v.to(dtype) for k, v in ref.state_dict().items()})
    ref.load_state_dict({k: v.float() for k, v in net.state_dict().items()})
    g = torch.Generator(device=DEV).manual_seed(1)
    x, y, gy = (torch.randn(B, n, D, generator=g, device=DEV).to(dtype).float() for n in (N, N - 1, N - 1))
    want = _run(ref, x, y, gy, 0, torch.float32)
    plain = _run(net, x, y, gy, 0, dtype)
    off = lambda r: [float((a.float() - w).norm() / (w.norm() + 1e-30)) for a, w in zip(r, want)]
    base = off(plain)
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    for rows in (16, 256, 4096):
        got = off(_run(net, x, y, gy, rows, dtype))
        # both round the same quantities to 16 bits (the chain rounds a few less): no further from the
        # fp32 module than the path with one GEMM per level, up to the scatter of single roundings
        for a, b in zip(got, base):
            assert a <= 1.25 * b + unit / 4, (rows, got, base)


def test_span_levels_bwd_refuses():
    lib = _lib.lib()
    z = torch.zeros(4096, device=DEV, dtype=torch.bfloat16)
    p = z.data_ptr()
    args = lambda Dh, dt, q=p: (p, q, p, p, p, p, 1, 2, 1, Dh, Dh, Dh, 3 * Dh, 3 * Dh, 3 * Dh, 3 * Dh, dt, 0)
    assert lib.hsa_span_levels_bwd(*args(48, 2)) == -95 and lib.hsa_span_levels_bwd(*args(64, 0)) == -95
    assert lib.hsa_span_levels_bwd(*args(64, 2, p + 2)) == -22
    torch.cuda.synchronize()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("case", [(2, 8, 3, 64), (1, 1, 2, 40), (3, 33, 1, 128)])
def test_strided_parent_backward(dtype, case):
    """hsa_build_parents_strided_bwd, and hsa_build_parents_level_bwd without a second gradient, on column
    slices of fused projections: the bits of the dense entry point, nothing written beside the slices."""
    import ctypes
    lib = _lib.lib()
    B, P, H, D = case
    Dm = H * D
    g = torch.Generator(device=DEV).manual_seed(P)
    mk = lambda rows, cols: torch.randn(B, rows, cols, generator=g, device=DEV).to(dtype)
    dout, qkv, kv = mk(P, Dm), mk(P, 3 * Dm), mk(2 * P, 2 * Dm)
    heads = lambda t: t.reshape(B, t.shape[1], H, D).contiguous()
    parts = [heads(dout)] + [heads(t) for t in qkv.split(Dm, dim=2)] + [heads(t) for t in kv.split(Dm, dim=2)]
    want = [torch.empty_like(parts[i]) for i in (1, 2, 3, 4, 5)]
    code, stream = _lib.dtype_code(dout), _lib.stream_of(dout)
    assert lib.hsa_build_parents_bwd(*(_lib.ptr(t) for t in parts + want), B, P, H, D, code, stream) == 0
    es = dout.element_size()
    A = ctypes.c_int64 * 11
    bs = A(P * Dm, *[3 * P * Dm] * 3, *[4 * P * Dm] * 2, *[3 * P * Dm] * 3, *[4 * P * Dm] * 2)
    rs = A(Dm, *[3 * Dm] * 3, *[2 * Dm] * 2, *[3 * Dm] * 3, *[2 * Dm] * 2)
    for name in ("hsa_build_parents_strided_bwd", "hsa_build_parents_level_bwd"):
        dqkv, dkv = torch.full_like(qkv, 7.0), torch.full_like(kv, 7.0)
        cols = lambda t, n: [t.data_ptr() + i * Dm * es for i in range(n)]
        first = [dout.data_ptr()] + ([None] if "level" in name else [])
        assert getattr(lib, name)(*first, *cols(qkv, 3), *cols(kv, 2), *cols(dqkv, 3), *cols(dkv, 2), B, P, H, D, bs, rs,
                                  code, stream) == 0
        got = [heads(t) for t in dqkv.split(Dm, dim=2)] + [heads(t) for t in dkv.split(Dm, dim=2)]
        assert all(torch.equal(a, b) for a, b in zip(got, want)), name
