"""Head sizes other than 32 / 64 / 128 channels on the 16-bit tile kernels: as precise as the gather kernels."""
import pytest
import torch

import oracle
import sparseattention_amd as sa
from sparseattention_amd.ops import functional as fn

pytestmark = pytest.mark.gpu
DEV = "cuda:0"


def _inputs(case, dtype, gscale=1.0):
    B, N, H, D, R = case
    g = torch.Generator().manual_seed(N + D)
    mk = lambda rows: torch.randn(B, rows, H, D, generator=g).to(dtype)
    return mk(N), mk(2 * N - 1), mk(2 * N - 1), (torch.randn(B, N, H, D, generator=g) * gscale).to(dtype)


def _autograd(q, k, v, go, R, causal):
    t = sa.build_tree_topology(q.shape[1], causal, device=DEV)
    leaves = [x.to(DEV).requires_grad_(True) for x in (q, k, v)]
    out = sa.hierarchical_attention(*leaves, t["forward_idx"], t["backward_gather"], t["forward_mask"] if causal else None, R)
    out.backward(go.to(DEV))
    return [out.detach()] + [x.grad for x in leaves]


def _gather(q, k, v, go, R, causal):
    t = sa.build_tree_topology(q.shape[1], causal, device=DEV)
    q, k, v, go = (x.to(DEV) for x in (q, k, v, go))
    out = fn.attention_forward(q, k, v, t["forward_idx"], t["forward_mask"] if causal else None, R, algo="gather")
    return [out] + list(fn.attention_backward(go, q, k, v, R, causal, algo="gather"))


# one size of every layout, one query block, strips of one and of four, both window variants
@pytest.mark.parametrize("case", [(2, 16, 2, 16, 5), (2, 256, 4, 48, 16), (1, 1024, 3, 80, 32), (2, 512, 4, 96, 16), (1, 128, 3, 120, 20)])
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("gscale", [1.0, 2.0 ** -10])
def test_no_less_precise_than_the_gather_kernels(case, causal, dtype, gscale):
    """Weights and the scores' gradients stay in fp32 in both directions.  Against fp64 the error is then
    that of rounding the result to 16 bits (2^-9, 2^-12 relative), to which fp32 sums of at most
    100 terms add less than 2^-17: no more than 1 % above the gather kernels' error, also for
    gradients near the smallest fp16 values."""
    q, k, v, go = _inputs(case, dtype, gscale)
    R = case[4]
    o = oracle.topology_tables(case[1], causal)
    ref = [x.double().requires_grad_(True) for x in (q, k, v)]
    want = oracle.attention_ref(*ref, o["forward_idx"], o["forward_mask"] if causal else None, R)
    want.backward(go.double())
    refs = [want.detach()] + [x.grad for x in ref]
    off = lambda res: [float((a.double().cpu() - w).norm() / w.norm()) for a, w in zip(res, refs)]
    got, base = off(_autograd(q, k, v, go, R, causal)), off(_gather(q, k, v, go, R, causal))
    for name, a, b in zip(("out", "dQ", "dK", "dV"), got, base):
        assert a <= 1.01 * b, (name, got, base)


def test_one_pass_backward_only_on_request():
    """The one-pass backward rounds the weights: such heads take it only where the caller asks for it."""
    case, R = (1, 128, 2, 96, 16), 16
    q, k, v, go = _inputs(case, torch.bfloat16)
    qd, kd, vd, gd = (x.to(DEV) for x in (q, k, v, go))
    two = fn.attention_backward(gd, qd, kd, vd, R, True)
    one = fn.attention_backward_saved(gd, qd, kd, vd, *fn.attention_forward_lse(qd, kd, vd, R, True), R, True)
    assert fn.one_pass_backward is None
    for mode, want in ((None, two), (True, one), (False, two)):
        fn.one_pass_backward = mode
        try:
            got = _autograd(q, k, v, go, R, True)[1:]
        finally:
            fn.one_pass_backward = None
        assert all(torch.equal(a, b) for a, b in zip(got, want)), mode
