"""Fused span levels at model widths of an odd number of 64 channels: contractions that are no multiple of the
kernels' rounds."""
import pytest
import torch

import sparseattention_amd as sa
from sparseattention_amd import _lib
from sparseattention_amd.ops import functional as fn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,C,H,Dh", [(1, 2, 1, 64), (2, 16, 2, 32), (2, 32, 3, 64), (3, 64, 5, 64), (1, 256, 11, 64), (4, 512, 7, 64),
                                      (2, 128, 10, 32), (1, 1024, 9, 64), (2, 64, 6, 32), (16, 512, 5, 64)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_levels_at_odd_widths(B, C, H, Dh, dtype):
    """A launch per wavefront and row tile, the weights staged per workgroup and the single launch round at the
    same places: same bits; and close to a product and a parent build per level."""
    dim = H * Dh
    assert dim % 128 == 64 and _lib.lib().hsa_cross_update_level_rows(B, H, Dh, 2) > 0
    g = torch.Generator().manual_seed(C + H + B)
    src = torch.randn(B, C, dim, generator=g).clamp(-1, 1).to(dtype).to(DEV)
    qkv = torch.randn(B, C - 1, 3 * dim, generator=g).clamp(-1, 1).to(dtype).to(DEV)
    w = (torch.randn(2 * dim, dim, generator=g) / dim ** 0.5).to(dtype).to(DEV)
    wp = fn.pack_kv_weights(w[:dim], w[dim:], H)
    lib, outs = _lib.lib(), []
    new = lambda: torch.empty(B, C - 1, dim, dtype=dtype, device=DEV)
    try:
        for min_tiles in (0, 1):
            assert lib.hsa_cross_update_level_tune(min_tiles, -1) == 0
            outs.append(fn.cross_update_top(src, qkv, wp, new(), H))
        if C <= fn.fused_top_rows(H, Dh, dtype):
            assert lib.hsa_cross_update_top_tune(1) == 0
            outs.append(fn.cross_update_top(src, qkv, wp, new(), H))
    finally:
        assert lib.hsa_cross_update_level_tune(8, -1) == 0 and lib.hsa_cross_update_top_tune(0) == 0
    assert all(torch.equal(outs[0], o) for o in outs[1:])
    cur, off, P, ref = src, 0, C // 2, []
    while P >= 1:
        kv = torch.nn.functional.linear(cur, w).view(B, 2 * P, 2, H, Dh)
        par = qkv[:, off:off + P].view(B, P, 3, H, Dh)
        o = torch.empty(B, P, H, Dh, dtype=dtype, device=DEV)
        fn.build_parents_strided(par[:, :, 0], par[:, :, 1], par[:, :, 2], kv[:, :, 0], kv[:, :, 1], out=o)
        cur = o.view(B, P, dim)
        ref.append(cur)
        off, P = off + P, P // 2
    # the same rounding points but for the order of the sums: single roundings that travel up the levels
    assert (outs[0].float() - torch.cat(ref, dim=1).float()).abs().max() < 2e-2


def test_widths_not_handled():
    for H, Dh in ((9, 32), (1, 32), (3, 24), (5, 48)):
        assert _lib.lib().hsa_cross_update_level_rows(1, H, Dh, 2) == 0


@pytest.mark.parametrize("B,N,H,Dh", [(2, 64, 5, 64), (3, 256, 3, 64), (1, 128, 10, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_module_at_odd_widths(B, N, H, Dh, dtype):
    """cross_update_Y without autograd (a chain of fused levels) and with it (a product per level), both against
    the module in fp32: the chain rounds the same quantities to 16 bits, or fewer."""
    torch.manual_seed(N)
    D = H * Dh
    net = sa.HierarchicalAttention(D, H, dropout=0.0).to(DEV).to(dtype)
    ref = sa.HierarchicalAttention(D, H, dropout=0.0).to(DEV)
    ref.load_state_dict({k: v.float() for k, v in net.state_dict().items()})
    g = torch.Generator(device=DEV).manual_seed(1)
    x, y = (torch.randn(B, n, D, generator=g, device=DEV).to(dtype) for n in (N, N - 1))
    with torch.no_grad():
        want, got = ref.cross_update_Y(x.float(), y.float()), net.cross_update_Y(x, y)
    plain = net.cross_update_Y(x.requires_grad_(True), y).detach()
    off = lambda t: float((t.float() - want).norm() / want.norm())
    unit = 2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -11
    assert off(got) <= 1.25 * off(plain) + unit / 4, (off(got), off(plain))
