"""Whole-tree build in one launch: head counts that are no power of two, heads that fill part of their lanes."""
import pytest
import torch

import oracle
import sparseattention_amd as sa
from sparseattention_amd import _lib

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


@pytest.fixture
def tree_knobs():
    def set_knobs(single_launch, threads):
        assert _lib.lib().hsa_build_tree_tune(single_launch, threads) == 0
    yield set_knobs
    assert _lib.lib().hsa_build_tree_tune(1, 0) == 0


# head groups of 4, 2 and 1; part heads on the specialised and on the general instantiation; both at once;
# one workgroup per batch element and several rounds of closing workgroups
@pytest.mark.parametrize("case", [(5, 1024, 12, 64), (3, 2048, 8, 96), (2, 256, 3, 48), (1, 4096, 7, 80), (2, 64, 6, 40),
                                  (2, 512, 5, 128), (1, 8192, 10, 72), (2, 16, 9, 64), (1, 128, 1, 96), (2, 8, 24, 32)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("threads", [0, 64, 256, 512])
def test_tree_single_launch_any_heads(case, dtype, threads, tree_knobs):
    B, N, H, D = case
    g = torch.Generator().manual_seed(N + H)
    qp, kp, vp = (torch.randn(B, N - 1, H, D, generator=g).to(dtype).to(DEV) for _ in range(3))
    # leaves and results as row slices of one buffer, the rows around the results kept
    kfull = torch.full((B, 2 * N + 1, H, D), 7.0, dtype=dtype, device=DEV)
    kfull[:, :N] = torch.randn(B, N, H, D, generator=g).to(dtype)
    vfull = kfull.clone()
    vfull[:, :N] = torch.randn(B, N, H, D, generator=g).to(dtype)
    kl, vl = kfull[:, :N], vfull[:, :N]
    tree_knobs(0, -1)
    stepwise = sa.build_tree(qp, kp, vp, kl, vl)
    tree_knobs(2, threads)
    for _ in range(2):  # the arrival counters are back at zero after a launch
        kfull[:, N:2 * N - 1] = vfull[:, N:2 * N - 1] = 0
        sa.build_tree(qp, kp, vp, kl, vl, out=kfull[:, N:2 * N - 1], out2=vfull[:, N:2 * N - 1])
        got = kfull[:, N:2 * N - 1]
        assert torch.equal(got, vfull[:, N:2 * N - 1])
        assert bool((kfull[:, 2 * N - 1:] == 7).all()) and bool((vfull[:, 2 * N - 1:] == 7).all())
        want = oracle.build_tree_ref(*(t.cpu() for t in (qp, kp, vp, kl, vl)), compute_dtype=torch.float64)
        err = (got.double().cpu() - want).abs()
        # bounds of the other tree tests: 1e-5 in fp32, 2e-2 + 1e-2 |ref| in 16 bits (one rounding per level)
        assert bool((err <= (1e-5 if dtype == torch.float32 else 2e-2 + 1e-2 * want.abs())).all())
        # same arithmetic in both paths: they may differ by the rounding of one fused multiply-add
        assert (got.float() - stepwise.float()).abs().max() <= (1e-6 if dtype == torch.float32 else 2e-2)


def test_tree_part_heads_with_infinite_keys(tree_knobs):
    """A key of -inf takes its weight away and nothing else, also in a head's last piece (which the lanes
    behind the head read again)."""
    B, N, H, D = 1, 16, 2, 24
    g = torch.Generator().manual_seed(1)
    qp = torch.rand(B, N - 1, H, D, generator=g).add_(0.5).to(torch.bfloat16).to(DEV)
    kp, vp = (torch.randn(B, N - 1, H, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    kl, vl = (torch.randn(B, N, H, D, generator=g).to(torch.bfloat16).to(DEV) for _ in range(2))
    kp[..., -1] = float("-inf")
    tree_knobs(0, -1)
    want = sa.build_tree(qp, kp, vp, kl, vl)
    tree_knobs(2, 64)
    got = sa.build_tree(qp, kp, vp, kl, vl)
    assert torch.isfinite(got).all() and (got.float() - want.float()).abs().max() <= 2e-2
