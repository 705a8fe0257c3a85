#!/usr/bin/env python3
"""Benchmark of the hierarchical sparse attention forward path on one MI355X.

A step = one pass of the hot path over one batch of synthetic input resident in HBM:
the bottom-up tree build (every BuildParentNodes level) that produces the node rows of
K_full / V_full, followed by the span attention forward.  Prints ONE JSON line.

  python bench.py [--gpus 1] [--steps K] [--warmup W] [--workload cfg3|cfg2|cfg5|cfg4]

The default run times the headline workload (cfg3) in full and, under `detail.configs`, the
other single-GPU configurations more briefly (kernel time, GB/s and fraction of the HBM peak of
the span attention and of the tree build, one-stream step time, CPU baseline of a bounded
sample each).
"""
import argparse
import ctypes
import json
import os
import sys
import time

ROOT = os.path.dirname(os.path.abspath(__file__))
if ROOT not in sys.path:
    sys.path.insert(0, ROOT)

WORKLOADS = {
    # name: (B, H, N, D, R, input scale, description)
    "cfg2": (16, 8, 512, 64, 8, 1.0 / 8, "B16 H8 N512 d64 bf16 SWA8 causal"),
    "cfg3": (8, 8, 2048, 64, 16, 1.0, "B8 H8 N2048 d64 bf16 SWA16 causal, parents built by the tree kernel"),
    "cfg5": (1, 16, 65536, 128, 32, 1.0, "B1 H16 N65536 d128 bf16 SWA32 causal"),
}
HBM_PEAK_GBS = 8000.0
E = 2  # bytes per element (bf16)


def parse():
    ap = argparse.ArgumentParser()
    ap.add_argument("--gpus", type=int, default=1)
    ap.add_argument("--steps", type=int, default=300)
    ap.add_argument("--warmup", type=int, default=30)
    ap.add_argument("--workload", default="cfg3", choices=sorted(WORKLOADS) + ["cfg4"])
    ap.add_argument("--noncausal", action="store_true")
    ap.add_argument("--seq-len", type=int, default=0, help="override the workload's N (a power of two)")
    ap.add_argument("--attention-only", action="store_true",
                    help="a step is the span attention alone, on span nodes drawn i.i.d. like the leaves "
                         "(isolates the attention kernel; the tree build is not run)")
    ap.add_argument("--sets", type=int, default=0,
                    help="buffer sets to rotate through (0 = enough that a step's data adds up to 1 GiB)")
    ap.add_argument("--streams", type=int, default=2,
                    help="HIP streams the steps alternate between (each step is an independent batch)")
    ap.add_argument("--no-cpu-baseline", action="store_true")
    ap.add_argument("--no-train-step", action="store_true",
                    help="cfg4: leave out the training step measured beside the forward (kernel profiles of the forward)")
    ap.add_argument("--cpu-seconds", type=float, default=12.0)
    ap.add_argument("--no-other-configs", action="store_true",
                    help="skip the brief measurements of the other configurations (detail.configs)")
    ap.add_argument("--calibrate-copy", action="store_true",
                    help="also launch a plain 64 MiB -> 64 MiB copy kernel 10 times (reference for HBM counters)")
    return ap.parse_args()


# ------------------------------------------------------------------------------------ CPU baseline
def host_threads():
    """Threads the CPU baseline uses: the cores this process may run on, capped by the
    OMP_NUM_THREADS the machine sets for its CPU share."""
    try:
        n = len(os.sched_getaffinity(0))
    except AttributeError:
        n = os.cpu_count() or 1
    if os.environ.get("OMP_NUM_THREADS", "").isdigit():
        n = min(n, int(os.environ["OMP_NUM_THREADS"]))
    return max(1, n)


def cpu_baseline(B, H, N, D, R, causal, scale, budget_s, with_plumbing=True):
    """Times the CPU restatement of the reference's PyTorch algorithm (tree build level by
    level + gather/einsum span attention) on this host's cores, bf16 tensors like the GPU run,
    on a bounded sample of the workload: at most two batch elements, and for long sequences a
    range of queries (the tree build is always timed whole)."""
    import torch
    import oracle
    cores = host_threads()
    torch.set_num_threads(cores)
    g = torch.Generator().manual_seed(0)
    bs = min(B, 2)
    mk = lambda rows: (torch.randn(bs, rows, H, D, generator=g) * scale).to(torch.bfloat16)
    q, kl, vl, qp, kp, vp = mk(N), mk(N), mk(N), mk(N - 1), mk(N - 1), mk(N - 1)
    t = oracle.topology_tables(N, causal)
    m = t["forward_mask"] if causal else None
    nq = min(N, 4096)  # queries of the sample

    def tree():
        tr = oracle.build_tree_ref(qp, kp, vp, kl, vl)
        return torch.cat([kl, tr], 1), torch.cat([vl, tr], 1)

    def attn(kf, vf):
        return oracle.attention_ref(q, kf, vf, t["forward_idx"], m, R, query_range=(N - nq, N))

    kf, vf = tree()
    attn(kf, vf)
    t_tree, t_attn, t_end = [], [], time.perf_counter() + budget_s
    while len(t_tree) < 2 or (time.perf_counter() < t_end and len(t_tree) < 30):
        t0 = time.perf_counter()
        kf, vf = tree()
        t1 = time.perf_counter()
        attn(kf, vf)
        t2 = time.perf_counter()
        t_tree.append(t1 - t0)
        t_attn.append(t2 - t1)
    med = lambda xs: sorted(xs)[len(xs) // 2]
    # seconds per head-query: the tree build covers bs*N*H of them, the attention sample bs*nq*H
    per_hq = med(t_tree) / (bs * N * H) + med(t_attn) / (bs * nq * H)
    res = {"value": 1.0 / per_hq, "unit": "head-queries/s", "cores": cores, "host_cpu_count": os.cpu_count(),
           "kind": "port",
           "sample": "%d of %d batch elements, tree build whole, span attention on %d of %d queries per element "
                     "(rate scaled per head-query); bf16, torch CPU, %d threads (the cores this process may use, "
                     "capped by OMP_NUM_THREADS), median of %d passes" % (bs, B, nq, N, cores, len(t_tree)),
           "tree_seconds_per_pass": med(t_tree), "attention_seconds_per_pass": med(t_attn)}
    if with_plumbing:
        res["cfg1_fp32"] = cpu_plumbing_case(oracle, cores)
    return res


def cpu_plumbing_case(oracle, cores):
    """The CPU-runnable configuration (B2 H4 N256 head 32, fp32, radius 8, causal and not): the CPU
    restatement timed in full and compared with the GPU kernel on the same seeded inputs."""
    import torch
    from sparseattention_amd.ops import functional as fn
    import sparseattention_amd as sa
    B, H, N, D, R = 2, 4, 256, 32, 8
    g = torch.Generator().manual_seed(0)
    q = torch.randn(B, N, H, D, generator=g)
    k = torch.randn(B, 2 * N - 1, H, D, generator=g)
    v = torch.randn(B, 2 * N - 1, H, D, generator=g)
    out = {"B": B, "H": H, "N": N, "D": D, "window_radius": R, "cores": cores}
    for causal in (True, False):
        t = oracle.topology_tables(N, causal)
        m = t["forward_mask"] if causal else None
        ts = []
        for _ in range(7):
            t0 = time.perf_counter()
            want = oracle.attention_ref(q, k, v, t["forward_idx"], m, R)
            ts.append(time.perf_counter() - t0)
        ts = sorted(ts[2:])  # two warm-ups, median of five
        td = sa.build_tree_topology(N, causal, device="cuda:0")
        got = fn.attention_forward(q.cuda(), k.cuda(), v.cuda(), td["forward_idx"],
                                   td["forward_mask"] if causal else None, R)
        tag = "causal" if causal else "noncausal"
        out[tag + "_cpu_head_queries_per_s"] = B * N * H / ts[len(ts) // 2]
        out[tag + "_gpu_vs_cpu_max_abs_err"] = (got.cpu() - want).abs().max().item()
    return out


# ------------------------------------------------------------------------------------ cfg4
LIB_LAUNCHERS = ("hsa_attn_fwd", "hsa_build_parents_fwd", "hsa_build_parents_strided_fwd", "hsa_cross_update_top_fwd",
                 "hsa_build_tree_fwd", "hsa_span_input_y", "hsa_topology_device", "hsa_cross_update_pack_weights")
# the same launches made from the native layer (csrc/torch_ops.cpp)
EXT_LAUNCHERS = ("span_attention", "build_tree", "add_layer_norm", "linear", "project", "query_key_value")


def lm_forward_measure(steps, warmup, train_step=True):
    """cfg4: forward of the 6-layer decoder LM (d_model 512, 8 heads, FFN 2048 GELU, vocab 50257,
    bf16, B=8, N=4096, window 16, random weights, token ids uniform over the vocabulary).  Returns
    the forward time, the share of the two module calls (event pairs around them) and the GPU time
    between event pairs put around every entry point of this library (its kernels alone)."""
    import torch
    import sparseattention_amd as sa
    from sparseattention_amd import _lib
    from sparseattention_amd.modules import attention as attn_mod

    dev = torch.device("cuda:0")
    B, N, V, d, H, ff, layers, R = 8, 4096, 50257, 512, 8, 2048, 6, 16
    torch.manual_seed(0)
    model = sa.TransformerLM(V, d, H, ff, layers, dropout=0.0, window_size=R, activation="gelu", max_len=N)
    model = model.to(dev).to(torch.bfloat16).eval()
    tok = torch.randint(0, V, (B, N), generator=torch.Generator().manual_seed(0)).to(dev)
    K = min(steps, 20)
    W = max(10, min(warmup, 20))  # the first forwards also grow the allocator's pools
    with torch.no_grad():
        for _ in range(W):
            model(tok)
        torch.cuda.synchronize()
        reps = []
        for _ in range(5):
            t0 = time.perf_counter()
            for _ in range(K):
                model(tok)
            torch.cuda.synchronize()
            reps.append((time.perf_counter() - t0) * 1e3 / K)
        ms = sorted(reps)[len(reps) // 2]
        # time share of the tree side (cross_update_Y: projections + one kernel per level) and of
        # the span attention op: the same forward with an event pair around each call
        spans = {"cross_update_Y": [], "hierarchical_attention": []}
        cls = attn_mod.HierarchicalAttention
        orig_c, orig_h = cls.cross_update_Y, attn_mod.hierarchical_attention

        def timed(store, f):
            def g(*a, **k):
                e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
                e0.record()
                r = f(*a, **k)
                e1.record()
                store.append((e0, e1))
                return r
            return g

        cls.cross_update_Y = timed(spans["cross_update_Y"], orig_c)
        attn_mod.hierarchical_attention = timed(spans["hierarchical_attention"], orig_h)
        model(tok)
        torch.cuda.synchronize()
        cls.cross_update_Y, attn_mod.hierarchical_attention = orig_c, orig_h

        # this library's launches alone: an event pair around every entry point that launches (layer by
        # layer through Python; the projections include the product that the library's rule leaves to hipBLASLt)
        native, sa.transformer.DecoderLayer._native = sa.transformer.DecoderLayer._native, lambda self, *a, **k: None
        handle = _lib.lib()
        own, saved = [], {}
        for owner, names in ((handle, LIB_LAUNCHERS), (_lib.ext(), EXT_LAUNCHERS)):
            for name in names:
                saved[owner, name] = getattr(owner, name)
                setattr(owner, name, timed(own, saved[owner, name]))
        model(tok)
        torch.cuda.synchronize()
        for (owner, name), f in saved.items():
            setattr(owner, name, f)
        sa.transformer.DecoderLayer._native = native

        # the same forward captured once into a HIP graph and replayed (no host work per launch);
        # a replay must reproduce the eager logits bit for bit, else the figure is not reported
        graph_ms = None
        eager = model(tok)
        side = torch.cuda.Stream()
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            model(tok)
        torch.cuda.current_stream().wait_stream(side)
        graph = torch.cuda.CUDAGraph()
        with torch.cuda.graph(graph):
            captured = model(tok)
        graph.replay()
        torch.cuda.synchronize()
        if torch.equal(captured, eager):
            t0 = time.perf_counter()
            for _ in range(K):
                graph.replay()
            torch.cuda.synchronize()
            graph_ms = (time.perf_counter() - t0) * 1e3 / K
            if not torch.equal(captured, eager):
                graph_ms = None
    share = {k: sum(a.elapsed_time(b) for a, b in v) for k, v in spans.items()}
    own_ms = sum(a.elapsed_time(b) for a, b in own)
    res = {"workload": "cfg4: decoder LM forward, 6L d512 h8 ffn2048 GELU vocab50257 bf16 B8 N4096 SWA16, random init, eval mode",
           "forward_ms": ms, "forward_ms_min": min(reps), "forward_ms_max": max(reps),
           "tokens_per_s": B * N / (ms * 1e-3), "steps": K, "warmup": W, "repetitions": len(reps),
           "ms_in_cross_update_Y_event_pairs": share["cross_update_Y"],
           "ms_in_hierarchical_attention_event_pairs": share["hierarchical_attention"],
           "share_cross_update_Y": share["cross_update_Y"] / ms,
           "share_hierarchical_attention": share["hierarchical_attention"] / ms,
           "ms_in_this_librarys_launches_event_pairs": own_ms, "launches_of_this_library": len(own),
           "hip_graph_replay_ms_per_forward": graph_ms,
           "calls_cross_update_Y": len(spans["cross_update_Y"]),
           "calls_hierarchical_attention": len(spans["hierarchical_attention"])}
    del eager, captured, graph
    torch.cuda.empty_cache()
    # one training step of the same model on the same batch (forward, cross-entropy on fp32 logits,
    # backward through this library's backward kernels, SGD update): reported beside the forward,
    # not part of `value`
    try:
        if not train_step:
            raise StopIteration
        model.train()
        tgt = torch.randint(0, V, (B, N), generator=torch.Generator().manual_seed(1)).to(dev)
        opt = torch.optim.SGD(model.parameters(), lr=1e-4)

        def train_step():
            opt.zero_grad(set_to_none=True)
            logits = model(tok)
            loss = torch.nn.functional.cross_entropy(logits.view(-1, V).float(), tgt.view(-1))
            loss.backward()
            opt.step()
            return loss

        for _ in range(3):
            last = train_step()
        torch.cuda.synchronize()
        tr = []
        for _ in range(3):
            t0 = time.perf_counter()
            for _ in range(4):
                last = train_step()
            torch.cuda.synchronize()
            tr.append((time.perf_counter() - t0) * 1e3 / 4)
        res["train_step_ms"] = sorted(tr)[1]
        res["train_tokens_per_s"] = B * N / (sorted(tr)[1] * 1e-3)
        res["train_loss_is_finite"] = bool(torch.isfinite(last).item())
        res["train_peak_memory_GB"] = torch.cuda.max_memory_allocated() / 1e9
        del opt, tgt, last
    except StopIteration:
        pass
    except Exception as exc:  # the forward figures stand on their own
        res["train_step_error"] = repr(exc)[:200]
    del model, tok
    torch.cuda.empty_cache()
    return res


def lm_forward_bench(args):
    r = lm_forward_measure(args.steps, args.warmup, not args.no_train_step)
    print(json.dumps({
        "metric": "LM forward tokens/sec, 6L d512 h8 ffn2048 GELU vocab50257 bf16 B8 N4096 SWA16",
        "value": r["tokens_per_s"], "unit": "tokens/s", "n_gpus": 1, "steps": r["steps"], "warmup": r["warmup"],
        "ms_per_step": r["forward_ms"], "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": r["workload"]}, "detail": r}))


# ------------------------------------------------------------------------------------ GPU side
class Hip:
    """The few runtime calls the timing needs (events that are attached to a dispatch)."""

    def __init__(self):
        self.lib = ctypes.CDLL("libamdhip64.so")
        self.lib.hipEventCreate.argtypes = [ctypes.POINTER(ctypes.c_void_p)]
        self.lib.hipEventDestroy.argtypes = [ctypes.c_void_p]
        self.lib.hipEventElapsedTime.argtypes = [ctypes.POINTER(ctypes.c_float), ctypes.c_void_p, ctypes.c_void_p]

    def event(self):
        ev = ctypes.c_void_p()
        assert self.lib.hipEventCreate(ctypes.byref(ev)) == 0
        return ev

    def free(self, ev):
        self.lib.hipEventDestroy(ev)

    def elapsed_ms(self, a, b):
        ms = ctypes.c_float()
        assert self.lib.hipEventElapsedTime(ctypes.byref(ms), a, b) == 0
        return ms.value


class Problem:
    """One workload's buffers in HBM (several sets, rotated so that no cache holds a step's data)
    and the argument tuples of the two entry points."""

    def __init__(self, torch, _lib, B, H, N, D, R, scale, causal, nsets, streams, iid_nodes=False):
        self.B, self.H, self.N, self.D, self.R, self.causal = B, H, N, D, R, causal
        self.L, self.M = N.bit_length() - 1, 2 * N - 1
        dev = torch.device("cuda:0")
        g = torch.Generator().manual_seed(0)
        M = self.M
        self.sets = []
        for _ in range(nsets):
            mk = lambda rows: (torch.randn(B, rows, H, D, generator=g) * scale).to(torch.bfloat16).to(dev)
            s = {"q": mk(N), "qp": mk(N - 1), "kp": mk(N - 1), "vp": mk(N - 1),
                 "kfull": torch.empty(B, M, H, D, dtype=torch.bfloat16, device=dev),
                 "vfull": torch.empty(B, M, H, D, dtype=torch.bfloat16, device=dev),
                 "out": torch.empty(B, N, H, D, dtype=torch.bfloat16, device=dev)}
            s["kfull"][:, :N] = mk(N)
            s["vfull"][:, :N] = mk(N)
            if iid_nodes:
                s["kfull"][:, N:] = mk(N - 1)
                s["vfull"][:, N:] = mk(N - 1)
            self.sets.append(s)
        torch.cuda.synchronize()
        P = lambda t: ctypes.c_void_p(t.data_ptr())
        node_off = N * H * D * E
        full_bs = M * H * D

        def tree_args(s, st):
            return (P(s["qp"]), P(s["kp"]), P(s["vp"]), P(s["kfull"]), P(s["vfull"]),
                    ctypes.c_void_p(s["kfull"].data_ptr() + node_off),
                    ctypes.c_void_p(s["vfull"].data_ptr() + node_off),
                    B, N, H, D, 0, 0, 0, full_bs, full_bs, full_bs, full_bs, _lib.HSA_BF16, st)

        def attn_args(s, st):
            return (P(s["q"]), P(s["kfull"]), P(s["vfull"]), None, None, P(s["out"]), None,
                    B, N, M, H, D, self.L, R, int(causal), _lib.HSA_BF16, _lib.ATTN_AUTO, st)

        self.tree_args, self.attn_args = tree_args, attn_args
        self.head_queries = B * N * H
        self.attn_bytes = E * B * H * D * (N + 2 * M + N)                         # Q + K_full + V_full + Out
        self.tree_bytes = E * B * H * D * (3 * (N - 1) + 2 * N + 2 * (N - 1))      # Qp,Kp,Vp + leaves + two copies out


def sets_for(step_bytes, requested, streams):
    n = requested or max(3, -(-(1 << 30) // step_bytes))
    while n % streams:
        n += 1
    return n


def step_bytes(B, H, N, D, attention_only):
    M = 2 * N - 1
    b = E * B * H * D * (N + 2 * M + N)
    if not attention_only:
        b += E * B * H * D * 3 * (N - 1)
    return b


def between_events(torch, stream, K, launch):
    """Average time of K calls of `launch(i)` between one pair of events on `stream`."""
    e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
    e0.record(stream)
    for i in range(K):
        launch(i)
    e1.record(stream)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / K


def kernel_times(torch, lib, hip, prob, stream, st, K, with_tree, reps=15):
    """Durations on one stream, inputs rotated as in the timed steps:
      b2b   K span-attention launches one after the other between one pair of events: the average
            launch duration (an upper bound of the kernel's own: the launch gaps are inside);
            repeated (see `repeated`), the median region counts;
      attn  the K steps once more with every attention dispatch carrying its own pair of HIP
            events (sorted); such a dispatch reads about 1 us longer than the same kernel in the
            rocprofv3 trace and than b2b;
      tree  K tree builds between one pair of events, repeated likewise."""
    n = len(prob.sets)
    targs = [prob.tree_args(s, st) for s in prob.sets]
    aargs = [prob.attn_args(s, st) for s in prob.sets]
    kev = [(hip.event(), hip.event()) for _ in range(K)]
    rc = 0
    for i in range(K):
        if with_tree:
            rc |= lib.hsa_build_tree_fwd(*targs[i % n])
        rc |= lib.hsa_attn_fwd_timed(*aargs[i % n], kev[i][0], kev[i][1])
    torch.cuda.synchronize()
    assert rc == 0, lib.hsa_last_error()
    attn = sorted(hip.elapsed_ms(a, b) for a, b in kev)
    for a, b in kev:
        hip.free(a)
        hip.free(b)
    b2b = repeated(lambda: between_events(torch, stream, K, lambda i: lib.hsa_attn_fwd(*aargs[i % n])), K,
                   min_reps=reps, min_total_ms=6.0)
    tree = None
    if with_tree:
        tree = repeated(lambda: between_events(torch, stream, K, lambda i: lib.hsa_build_tree_fwd(*targs[i % n])), K,
                        min_reps=reps, min_total_ms=6.0)
    return {"attn": attn, "b2b": median(b2b), "tree": median(tree) if tree else None,
            "b2b_samples": b2b, "tree_samples": tree}


def wall_ms_per_step(torch, lib, prob, st_list, K, with_tree):
    """K steps between two synchronisations, set i on stream i mod len(st_list)."""
    n, ns = len(prob.sets), len(st_list)
    targs = [prob.tree_args(s, st_list[i % ns]) for i, s in enumerate(prob.sets)]
    aargs = [prob.attn_args(s, st_list[i % ns]) for i, s in enumerate(prob.sets)]
    torch.cuda.synchronize()
    t0 = time.perf_counter()
    rc = 0
    for i in range(K):
        if with_tree:
            rc |= lib.hsa_build_tree_fwd(*targs[i % n])
        rc |= lib.hsa_attn_fwd(*aargs[i % n])
    torch.cuda.synchronize()
    t1 = time.perf_counter()
    assert rc == 0, lib.hsa_last_error()
    return (t1 - t0) * 1e3 / K


def repeated(measure, K, min_reps=15, min_total_ms=12.0, max_reps=400):
    """`measure()` times one region of K steps and returns ms per step.  Runs it at least
    `min_reps` times and until the regions add up to `min_total_ms` of work, so that the figure
    does not rest on a single sub-millisecond sample whatever K is; returns the sorted samples."""
    xs = [measure()]
    need = max(min_reps, int(min_total_ms / max(xs[0] * K, 1e-6)) + 1)
    for _ in range(min(need, max_reps) - 1):
        xs.append(measure())
    return sorted(xs)


def median(xs):
    return xs[len(xs) // 2]


def copy_reference(torch, stream, K, nbytes):
    """Average duration (ms) of torch's device-to-device copy that moves `nbytes` in all (half read,
    half written), buffers rotated through 1 GiB, K copies between one pair of events; and the
    bytes it moved."""
    dev = torch.device("cuda", torch.cuda.current_device())
    half = nbytes // 2 // 2 * 2
    ncopy = max(3, -(-(1 << 30) // (2 * half)))
    csrc = [torch.empty(half // 2, device=dev, dtype=torch.bfloat16).normal_() for _ in range(ncopy)]
    cdst = [torch.empty(half // 2, device=dev, dtype=torch.bfloat16) for _ in range(ncopy)]
    with torch.cuda.stream(stream):
        for i in range(min(K, 2 * ncopy)):
            cdst[i % ncopy].copy_(csrc[i % ncopy])
        e0, e1 = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
        e0.record(stream)
        for i in range(K):
            cdst[i % ncopy].copy_(csrc[i % ncopy])
        e1.record(stream)
    torch.cuda.synchronize()
    return e0.elapsed_time(e1) / K, 2 * half


def backward_times(torch, _lib, lib, prob, stream, st, K, causal):
    """Average time of the span attention backward on the problem's rotated inputs, both
    launches of each formulation between one pair of events: (two passes, one pass on the saved
    forward state or None where that is not built)."""
    B, H, N, D, R = prob.B, prob.H, prob.N, prob.D, prob.R
    M, L = 2 * N - 1, N.bit_length() - 1
    dev = prob.sets[0]["q"].device
    nsets = len(prob.sets)
    P = lambda t: ctypes.c_void_p(t.data_ptr())
    s0 = prob.sets[0]
    gq = torch.randn(B, N, H, D, device=dev).to(torch.bfloat16)
    dq_, dk_, dv_ = torch.empty_like(gq), torch.empty_like(s0["kfull"]), torch.empty_like(s0["kfull"])
    wsb = int(lib.hsa_attn_bwd_workspace_bytes(B, N, M, H, D, L, R, _lib.HSA_BF16, _lib.ATTN_AUTO))
    wsp = torch.empty(max(wsb, 4) // 4 + 1, device=dev, dtype=torch.float32)
    bargs = [(P(s["q"]), P(s["kfull"]), P(s["vfull"]), P(gq), P(dq_), P(dk_), P(dv_), P(wsp), wsp.numel() * 4,
              B, N, M, H, D, L, R, int(causal), _lib.HSA_BF16, _lib.ATTN_AUTO, st) for s in prob.sets]
    for i in range(3):
        assert lib.hsa_attn_bwd(*bargs[i % nsets]) == 0, lib.hsa_last_error()
    two_ms = median(repeated(
        lambda: between_events(torch, stream, K, lambda i: lib.hsa_attn_bwd(*bargs[i % nsets])), K, min_reps=7,
        min_total_ms=6.0))
    # the one-pass backward on saved forward state, where it is built
    one_ms = None
    if int(lib.hsa_attn_bwd_saved_workspace_bytes(B, N, M, H, D, L, R, int(causal), _lib.HSA_BF16)) > 0:
        saved = []
        for s in prob.sets:
            o_ = torch.empty_like(s["q"])
            lse_ = torch.empty(B, N, H, device=dev, dtype=torch.float32)
            assert lib.hsa_attn_fwd_lse(P(s["q"]), P(s["kfull"]), P(s["vfull"]), P(o_), P(lse_), B, N, M, H, D, L, R,
                                        int(causal), _lib.HSA_BF16, st) == 0, lib.hsa_last_error()
            saved.append((o_, lse_))
        b1args = [(P(s["q"]), P(s["kfull"]), P(s["vfull"]), P(o_), P(lse_), P(gq), P(dq_), P(dk_), P(dv_), P(wsp),
                   wsp.numel() * 4, B, N, M, H, D, L, R, int(causal), _lib.HSA_BF16, st)
                  for s, (o_, lse_) in zip(prob.sets, saved)]
        for i in range(3):
            assert lib.hsa_attn_bwd_saved(*b1args[i % nsets]) == 0, lib.hsa_last_error()
        one_ms = median(repeated(
            lambda: between_events(torch, stream, K, lambda i: lib.hsa_attn_bwd_saved(*b1args[i % nsets])), K,
            min_reps=7, min_total_ms=6.0))
    return two_ms, one_ms


def brief_config(torch, _lib, lib, hip, name, causal, K, cpu_seconds):
    """Kernel times, GB/s and fraction of the HBM peak of one configuration, its one-stream step
    time, and its CPU baseline on a bounded sample."""
    B, H, N, D, R, scale, desc = WORKLOADS[name]
    stream = torch.cuda.current_stream()
    st = ctypes.c_void_p(stream.cuda_stream)
    nsets = sets_for(step_bytes(B, H, N, D, False), 0, 1)
    prob = Problem(torch, _lib, B, H, N, D, R, scale, causal, nsets, 1)
    for _ in range(2):
        wall_ms_per_step(torch, lib, prob, [st], min(K, 10), True)
    step_ms = median(repeated(lambda: wall_ms_per_step(torch, lib, prob, [st], K, True), K, min_reps=7, min_total_ms=6.0))
    kt = kernel_times(torch, lib, hip, prob, stream, st, K, True, reps=7)
    attn, tree_ms, a_ms = kt["attn"], kt["tree"], kt["b2b"]
    e_ms = sum(attn) / len(attn)
    rec = {"workload": desc if causal else desc.replace("causal", "not causal"),
           "head_queries_per_step": prob.head_queries, "buffer_sets_rotated": nsets, "steps": K,
           "attn_back_to_back_avg_ms": a_ms, "attn_in_step_dispatch_event_avg_ms": e_ms,
           "attn_in_step_dispatch_event_median_ms": attn[len(attn) // 2],
           "attn_algorithmic_bytes": prob.attn_bytes,
           "attn_GBps": prob.attn_bytes / (a_ms * 1e-3) / 1e9,
           "attn_frac_of_hbm_peak": prob.attn_bytes / (a_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
           "attn_frac_of_hbm_peak_in_step_events": prob.attn_bytes / (e_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
           "tree_build_avg_launch_ms": tree_ms, "tree_algorithmic_bytes": prob.tree_bytes,
           "tree_GBps": prob.tree_bytes / (tree_ms * 1e-3) / 1e9,
           "tree_frac_of_hbm_peak": prob.tree_bytes / (tree_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
           "single_stream_ms_per_step": step_ms,
           "single_stream_head_queries_per_s": prob.head_queries / (step_ms * 1e-3),
           "device_copy_of_attn_bytes_ms": copy_reference(torch, stream, K, prob.attn_bytes)[0],
           "device_copy_of_tree_bytes_ms": copy_reference(torch, stream, K, prob.tree_bytes)[0]}
    two_ms, one_ms = backward_times(torch, _lib, lib, prob, stream, st, K, causal)
    bwd_bytes = 2 * B * H * D * (3 * N + 4 * (2 * N - 1))  # Q, dO, dQ and K, V, dK, dV once each
    rec["attn_backward_avg_ms"] = two_ms
    rec["attn_backward_one_pass_avg_ms"] = one_ms
    rec["attn_backward_algorithmic_bytes"] = bwd_bytes
    best = min(two_ms, one_ms) if one_ms is not None else two_ms
    rec["attn_backward_frac_of_hbm_peak"] = bwd_bytes / (best * 1e-3) / 1e9 / HBM_PEAK_GBS
    del prob
    torch.cuda.empty_cache()
    if cpu_seconds > 0:
        rec["cpu_baseline"] = cpu_baseline(B, H, N, D, R, causal, scale, cpu_seconds, with_plumbing=False)
    return rec


def main():
    args = parse()
    if args.gpus != 1:
        print("bench.py measures one GPU only: this build has no multi-GPU path (every (batch, head) is "
              "independent, so the path would shard over batch or heads without any exchange). "
              "Re-run with --gpus 1.", file=sys.stderr)
        sys.exit(2)
    import torch
    from sparseattention_amd import _lib

    if args.workload == "cfg4":
        return lm_forward_bench(args)
    B, H, N, D, R, scale, desc = WORKLOADS[args.workload]
    if args.seq_len:
        assert args.seq_len >= 64 and args.seq_len & (args.seq_len - 1) == 0, "--seq-len must be a power of two >= 64"
        desc = desc.replace("N%d" % N, "N%d" % args.seq_len)
        N = args.seq_len
    causal = not args.noncausal
    if not causal:
        desc = desc.replace("causal", "not causal")
    if args.attention_only:
        desc = desc.replace(", parents built by the tree kernel", ", span nodes drawn i.i.d.")
    dev = torch.device("cuda:0")
    torch.cuda.set_device(dev)
    lib = _lib.lib()
    hip = Hip()
    K = args.steps
    with_tree = not args.attention_only

    stream = torch.cuda.current_stream(dev)
    st = ctypes.c_void_p(stream.cuda_stream)
    # Steps are independent batches: they alternate between `--streams` HIP streams (default
    # priority), so one step's launch ramps and tails overlap the next step's streaming kernels.
    # A buffer set always goes to the same stream, so two steps that touch the same buffers are
    # ordered.  Enough sets are rotated that the data of consecutive steps adds up to 1 GiB,
    # four times the 256 MB Infinity Cache (with 4 x 100 MB the attention alone measured 10 %
    # faster than with 8 or 16 sets: part of it was served from that cache).
    nstreams = max(1, args.streams)
    sbytes = step_bytes(B, H, N, D, args.attention_only)
    nsets = sets_for(sbytes, args.sets, nstreams)
    side = [torch.cuda.Stream(device=dev) for _ in range(nstreams)] if nstreams > 1 else [stream]
    side_st = [ctypes.c_void_p(x.cuda_stream) for x in side]
    prob = Problem(torch, _lib, B, H, N, D, R, scale, causal, nsets, nstreams, iid_nodes=args.attention_only)
    L, M = prob.L, prob.M
    assert lib.hsa_attn_fwd_uses_tile(N, M, H, D, L, R, _lib.HSA_BF16, 1, 0) == 1

    for _ in range(max(1, args.warmup // max(1, nsets))):
        wall_ms_per_step(torch, lib, prob, side_st, nsets, with_tree)

    # --- timed region: exactly K steps between two synchronisations -----------------------
    #     The region is repeated (at least 15 times, and until 12 ms of work have been timed) and
    #     the median region is reported: with --steps 20 a single region is 0.8 ms of work, and
    #     one scheduler hiccup would move the figure by several per cent.
    step_samples = repeated(lambda: wall_ms_per_step(torch, lib, prob, side_st, K, with_tree), K)
    ms_per_step = median(step_samples)

    # --- the same K steps one after the other on a single stream (the latency of a step) ----
    wall_ms_per_step(torch, lib, prob, [st], min(args.warmup, 10), with_tree)
    serial_samples = repeated(lambda: wall_ms_per_step(torch, lib, prob, [st], K, with_tree), K)
    serial_ms_per_step = median(serial_samples)

    # --- duration of the dominant kernel, on one stream with the same rotation of inputs: K
    #     attention launches between one pair of events (the figure of the roofline object), the
    #     K steps once more with an event pair on every attention dispatch (kept out of the timed
    #     region: such a dispatch costs the step about 3 us of completion handling), K tree
    #     builds and K whole steps between one pair of events each ------------------------------
    kt = kernel_times(torch, lib, hip, prob, stream, st, K, with_tree)
    attn_kernel_ms, tree_b2b_ms, attn_b2b_ms = kt["attn"], kt["tree"], kt["b2b"]
    attn_avg_ms = attn_b2b_ms
    attn_event_avg_ms = sum(attn_kernel_ms) / K

    # --- backward of the span attention (next-row kernel), same rotation of inputs ----------------
    attn_bwd_ms, attn_bwd1_ms = backward_times(torch, _lib, lib, prob, stream, st, K, causal)

    # --- reference point: a plain device-to-device copy that moves as many bytes as one launch of
    #     the attention kernel (half read, half written), buffers rotated through 1 GiB like the
    #     inputs above, K copies between one pair of events ---------------------------------------
    copy_ms, copy_bytes = copy_reference(torch, stream, K, prob.attn_bytes)
    tree_copy_ms = copy_reference(torch, stream, K, prob.tree_bytes)[0] if with_tree else None

    if args.calibrate_copy:
        n = 64 * 2**20 // 2
        src = [torch.randn(n, device=dev).to(torch.bfloat16) for _ in range(5)]
        dst = [torch.empty(n, device=dev, dtype=torch.bfloat16) for _ in range(5)]
        for i in range(10):
            dst[i % 5].copy_(src[i % 5])
        torch.cuda.synchronize()

    # HBM bytes per launch of the attention kernel as counted by rocprofv3 --pmc FETCH_SIZE /
    # WRITE_SIZE (scaled by a plain copy of known size); recorded under profiles/
    traffic = None
    tpath = os.path.join(ROOT, "profiles", "attn_tile_%s_traffic.json" % args.workload)
    if os.path.exists(tpath):
        rec = json.load(open(tpath))
        if rec.get("causal") == causal and not args.seq_len:
            traffic = rec["traffic_bytes_per_launch"]

    head_queries, attn_bytes, tree_bytes = prob.head_queries, prob.attn_bytes, prob.tree_bytes
    achieved = attn_bytes / (attn_avg_ms * 1e-3) / 1e9
    step_algorithmic = attn_bytes + (tree_bytes if with_tree else 0)
    result = {
        "metric": "attn fwd queries/sec + % HBM roofline, B8 H8 N2048 d64 bf16 SWA16",
        "value": head_queries / (ms_per_step * 1e-3),
        "unit": "head-queries/s",
        "n_gpus": 1, "steps": K, "warmup": args.warmup, "ms_per_step": ms_per_step,
        "higher_is_better": True, "scaling": "weak", "vs_baseline": None,
        "dtype": "bf16", "data": "synthetic",
        "config": {"workload": "%s: %s; step = tree build + span attention forward on one batch; independent batches alternate between %d HIP streams" % (args.workload, desc, nstreams),
                   "B": B, "H": H, "N": N, "D": D, "window_radius": R, "causal": causal,
                   "buffer_sets_rotated": nsets, "bytes_per_set": E * B * H * D * (N + 2 * M + N + 3 * (N - 1)), "streams": nstreams},
        "roofline": {"bound": "hbm", "kernel": "attn_tile_kernel (span attention forward)",
                     "achieved": achieved, "peak": HBM_PEAK_GBS, "unit": "GB/s",
                     "frac": achieved / HBM_PEAK_GBS, "traffic": traffic,
                     "algorithmic_bytes_per_launch": attn_bytes, "avg_launch_ms": attn_avg_ms,
                     "timing": "K launches of the kernel one after the other on one stream between one pair of HIP events, inputs rotated as in the timed steps (launch gaps included: an upper bound of the kernel's duration)",
                     "per_dispatch_events": {"avg_ms": attn_event_avg_ms, "median_ms": attn_kernel_ms[K // 2],
                                             "min_ms": attn_kernel_ms[0],
                                             "frac": attn_bytes / (attn_event_avg_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                                             "timing": "the K steps once more, one stream, a HIP event pair attached to every attention dispatch (reads about 1 us more than the same dispatch in the rocprofv3 kernel trace)"}},
        "detail": {"timed_regions": {"regions_of_K_steps": len(step_samples), "reported": "median region",
                                     "ms_per_step_min": step_samples[0], "ms_per_step_max": step_samples[-1],
                                     "single_stream_ms_per_step_min": serial_samples[0],
                                     "single_stream_ms_per_step_max": serial_samples[-1],
                                     "attn_launch_ms_min": kt["b2b_samples"][0], "attn_launch_ms_max": kt["b2b_samples"][-1]},
                   "single_stream_ms_per_step": serial_ms_per_step,
                   "single_stream_head_queries_per_s": head_queries / (serial_ms_per_step * 1e-3),
                   "step_algorithmic_bytes": step_algorithmic,
                   "step_GBps_two_streams": step_algorithmic / (ms_per_step * 1e-3) / 1e9,
                   "step_frac_of_hbm_peak_two_streams": step_algorithmic / (ms_per_step * 1e-3) / 1e9 / HBM_PEAK_GBS,
                   "attn_only_head_queries_per_s": head_queries / (attn_avg_ms * 1e-3),
                   "attn_backward_avg_ms": attn_bwd_ms,
                   "attn_backward_one_pass_avg_ms": attn_bwd1_ms,
                   "attn_backward_algorithmic_bytes": E * B * H * D * (2 * N + 2 * M + N + 2 * M),
                   "attn_backward_frac_of_hbm_peak": E * B * H * D * (2 * N + 2 * M + N + 2 * M) / (
                       min(attn_bwd_ms, attn_bwd1_ms or attn_bwd_ms) * 1e-3) / 1e9 / HBM_PEAK_GBS,
                   "device_copy_of_the_same_bytes": {
                       "bytes": copy_bytes, "avg_ms": copy_ms, "GBps": copy_bytes / (copy_ms * 1e-3) / 1e9,
                       "frac_of_hbm_peak": copy_bytes / (copy_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
                       "attention_kernel_vs_copy": copy_ms / attn_avg_ms,
                       "note": "torch's device-to-device copy of as many bytes as one attention launch moves (half read, half written), buffers rotated through 1 GiB, K copies between one pair of events: what a kernel without arithmetic reaches on this GPU"}},
    }
    if with_tree:
        result["roofline_tree"] = {
            "bound": "hbm", "kernel": "build_tree_fused_kernel (hsa_build_tree_fwd, every level, one launch)",
            "achieved": tree_bytes / (tree_b2b_ms * 1e-3) / 1e9, "peak": HBM_PEAK_GBS, "unit": "GB/s",
            "frac": tree_bytes / (tree_b2b_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
            "algorithmic_bytes_per_launch": tree_bytes, "avg_launch_ms": tree_b2b_ms,
            "timing": "K calls between one pair of events on the launch stream (includes the gaps between launches)",
            "device_copy_of_the_same_bytes_ms": tree_copy_ms}
        result["detail"]["tree_build_avg_launch_ms"] = tree_b2b_ms
        result["detail"]["tree_algorithmic_bytes"] = tree_bytes
        result["detail"]["tree_GBps"] = tree_bytes / (tree_b2b_ms * 1e-3) / 1e9
    del prob
    torch.cuda.empty_cache()

    headline = args.workload == "cfg3" and causal and not args.seq_len and not args.attention_only
    if headline and not args.no_other_configs:
        # the quantity the 60 % target is stated on, timed on the wall clock: the attention alone,
        # one stream, span nodes drawn i.i.d., enough sets that a pass over them is 1 GiB
        ns = sets_for(step_bytes(B, H, N, D, True), 0, 1)
        ao = Problem(torch, _lib, B, H, N, D, R, scale, causal, ns, 1, iid_nodes=True)
        wall_ms_per_step(torch, lib, ao, [st], 20, False)
        ao_ms = median(repeated(lambda: wall_ms_per_step(torch, lib, ao, [st], K, False), K, min_reps=7, min_total_ms=6.0))
        ao_k = kernel_times(torch, lib, hip, ao, stream, st, K, False)
        result["detail"]["attention_only_one_stream"] = {
            "ms_per_launch_wall_clock": ao_ms, "head_queries_per_s_wall_clock": head_queries / (ao_ms * 1e-3),
            "frac_of_hbm_peak_wall_clock": attn_bytes / (ao_ms * 1e-3) / 1e9 / HBM_PEAK_GBS,
            "kernel_avg_ms_between_events": ao_k["b2b"], "dispatch_event_avg_ms": sum(ao_k["attn"]) / K,
            "buffer_sets_rotated": ns}
        del ao
        torch.cuda.empty_cache()
        kb = min(K, 60)
        cs = 0.0 if args.no_cpu_baseline else max(4.0, args.cpu_seconds / 2)
        result["detail"]["configs"] = {
            "cfg2": brief_config(torch, _lib, lib, hip, "cfg2", True, kb, cs),
            "cfg3_noncausal": brief_config(torch, _lib, lib, hip, "cfg3", False, kb, 0.0),
            "cfg5": brief_config(torch, _lib, lib, hip, "cfg5", True, min(kb, 20), cs),
        }
        # the decoder LM (its own metric: tokens/s of the forward; see --workload cfg4)
        result["detail"]["configs"]["cfg4"] = lm_forward_measure(20, 10, not args.no_train_step)
    if not args.no_cpu_baseline:
        result["cpu_baseline"] = cpu_baseline(B, H, N, D, R, causal, scale, args.cpu_seconds)
    if args.attention_only:
        result["config"]["workload"] = result["config"]["workload"].replace(
            "step = tree build + span attention forward", "step = span attention forward alone (i.i.d. span nodes)")
    if not headline:
        result["metric"] = "attn fwd queries/sec + % HBM roofline, " + desc
    print(json.dumps(result))


if __name__ == "__main__":
    main()
