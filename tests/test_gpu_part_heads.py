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


def _same(got, want, atol, what, kinds=True):
    """Infinities and NaN in the same places (kinds: and the same ones), everything else within atol."""
    got, want = got.float(), want.float()
    odd = ~torch.isfinite(want)
    assert torch.equal(~torch.isfinite(got), odd), what
    assert not kinds or torch.equal(torch.nan_to_num(got[odd], 0.0, 1.0, -1.0), torch.nan_to_num(want[odd], 0.0, 1.0, -1.0)), what
    if not bool(odd.all()):
        assert (got[~odd] - want[~odd]).abs().max() <= atol, (what, float((got[~odd] - want[~odd]).abs().max()))


# heads that end inside a contraction step and heads that fill it, layouts of 32, 64 and 128 channels
ODD_SIZES = [(1, 16, 2, 16, 3), (1, 32, 2, 24, 5), (2, 64, 2, 48, 16), (1, 256, 2, 80, 20), (1, 128, 3, 96, 16)]


@pytest.mark.parametrize("case", ODD_SIZES)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinite_keys_and_values(case, causal, dtype):
    """Infinities and NaN reach the queries that attend to their row and no others, and a key of -inf takes its
    weight away and nothing else: what the gather kernels give, element by element."""
    B, N, H, D, R = case
    t = sa.build_tree_topology(N, causal, device=DEV)
    mask = t["forward_mask"] if causal else None
    inf, nan = float("inf"), float("nan")

    def check(what, edit):
        q, k, v, _ = (x.to(DEV) for x in _inputs(case, dtype))
        q = q.abs() + 0.5
        edit(q, k, v)
        run = lambda algo: fn.attention_forward(q, k, v, t["forward_idx"], mask, R, algo=algo)
        want = run("gather")
        # fp32 sums in another order, then one rounding: one unit of the last place of results up to 4.
        # (At 16 channels the gather kernel multiplies dead slots' zeros with the query's own value row.)
        _same(run("tile"), want, 2 ** -6 if dtype == torch.bfloat16 else 2 ** -9, what, kinds=D != 16)

    def keys_gone(q, k, v):
        k[:, N // 2, :, -1] = -inf        # a leaf, in the head's last channel
        k[:, N, 0, 0] = -inf              # nodes of the first level and of the level below the root
        k[:, 2 * N - 3, :, -1] = -inf

    def all_keys_gone(q, k, v):
        k[:, :, -1] = -inf                # every key of one head

    def odd_row(value):
        def edit(q, k, v):
            k[:, N // 2 + 3, 0, 1] = value
            v[:, N // 2 + 3, -1, 2] = value
            v[:, 2 * N - 2] = value       # the root: nobody attends to it
            k[:, 2 * N - 2] = value
        return edit

    def odd_query(q, k, v):
        q[:, 5, 0, 3] = inf
        q[:, 7, -1, 0] = nan

    check("keys of -inf", keys_gone)
    check("all keys of -inf", all_keys_gone)
    for value in (inf, -inf, nan):
        check("a row with %s" % value, odd_row(value))
    check("queries", odd_query)


@pytest.mark.parametrize("case", ODD_SIZES)
@pytest.mark.parametrize("causal", [True, False])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
def test_infinities_in_the_backward(case, causal, dtype):
    """Gradients stay finite wherever the gather kernels' are: an infinity or a NaN does not reach rows
    that its row has nothing to do with."""
    B, N, H, D, R = case
    inf, nan = float("inf"), float("nan")

    def check(what, edit, rows_of_dv=True):
        q, k, v, go = (x.to(DEV) for x in _inputs(case, dtype))
        q = q.abs() + 0.5
        edit(q, k, v, go)
        want = fn.attention_backward(go, q, k, v, R, causal, algo="gather")
        got = fn.attention_backward(go, q, k, v, R, causal, algo="tile")
        for name, a, b in zip(("dQ", "dK", "dV"), got, want):
            a, b = a.float(), b.float()
            ok = torch.isfinite(b)
            if name == "dV" and not rows_of_dv:  # a row of dO counts as a whole there
                ok = ok.all(dim=-1, keepdim=True).expand_as(ok)
            # (a NaN score leaves the query's sum of weights at its lower bound of 1e-5, in both: the other keys
            # then get 1e5 times their share, which says nothing)
            ok = ok & (torch.where(ok, b, 0).abs().amax(dim=-1, keepdim=True) < 1e3)
            assert bool(torch.isfinite(a[ok]).all()), (what, name)
            # up to 64 + 22 terms of size 4 summed in fp32 and rounded once: a unit of the last place of
            # values up to 64 (bf16: 2^-2), which the largest sums here stay below
            if bool(ok.any()):
                bound = (2 ** -8 if dtype == torch.bfloat16 else 2 ** -11) * (b[ok].abs() + 1.0)
                assert bool(((a[ok] - b[ok]).abs() <= 2 * bound).all()), (what, name)

    def keys_gone(q, k, v, go):
        k[:, N // 2, :, -1] = -inf
        k[:, N, 0, 0] = -inf

    def odd_row(value):
        def edit(q, k, v, go):
            k[:, N // 2 + 3, 0, 1] = value
            v[:, N // 2 + 5, -1, 2] = value
            v[:, 2 * N - 2] = value
            k[:, 2 * N - 2] = value
        return edit

    def odd_query(q, k, v, go):
        q[:, 5, 0, 3] = nan

    def odd_gradient(q, k, v, go):
        go[:, 9, 0, 3] = inf

    check("keys of -inf", keys_gone)
    for value in (inf, nan):
        check("a row with %s" % value, odd_row(value))
    check("a query", odd_query)
    check("a row of dO", odd_gradient, rows_of_dv=False)
    # every key of one head: no weights, so no gradients
    q, k, v, go = (x.to(DEV) for x in _inputs(case, dtype))
    q, k[:, :, 0] = q.abs() + 0.5, -inf
    dq, dk, dv = fn.attention_backward(go, q, k, v, R, causal, algo="tile")
    assert not dq[:, :, 0].any() and not dk[:, :, 0].any() and not dv[:, :, 0].any()
    assert all(bool(torch.isfinite(x[:, :, 1:]).all()) for x in (dq, dk, dv))


@pytest.mark.parametrize("D", [24, 48, 72, 120])
def test_infinite_keys_in_the_one_pass_backward(D):
    """A key of -inf in the head's last channel takes its weight away there too.  (dQ gets 0 times the key.)"""
    case, R = (1, 128, 2, D, 16), 16
    q, k, v, go = (x.to(DEV) for x in _inputs(case, torch.bfloat16))
    q = q.abs() + 0.5
    k[:, 64, :, -1] = k[:, 128, :, -1] = -float("inf")
    out, lse = fn.attention_forward_lse(q, k, v, R, True)
    assert bool(torch.isfinite(out).all()) and bool(torch.isfinite(lse).all())
    one = fn.attention_backward_saved(go, q, k, v, out, lse, R, True)
    two = fn.attention_backward(go, q, k, v, R, True)
    for a, b in zip(one[1:], two[1:]):
        assert bool(torch.isfinite(a).all())
        # weights and score gradients rounded to 8 bits, delta from rounded outputs: 2^-9 each, a few of them
        assert (a.float() - b.float()).norm() <= 2e-2 * b.float().norm()
