"""`HierarchicalAttention`: the nn.Module around the two ops.

Parameter names, shapes and method signatures follow the reference's
hierarchical_attention/modules/attention.py:10-270 so that its state dicts load
unchanged; the dense projections are `nn.Linear` modules whose products run on this package's kernels where
they are the faster ones (`ops/linear.py`), the tree build and the span attention are the HIP kernels.
"""
from __future__ import annotations

import ctypes
import math
from typing import List, Optional

import torch
import torch.nn as nn
import torch.nn.functional as F

from .. import _lib
from ..ops.functional import build_parent_nodes, hierarchical_attention, pack_kv_weights
from ..ops.linear import FORWARDS, linear, project, query_key_value, query_key_value_rows, weight_and_bias
from ..ops.topology import build_tree_topology


def _level_sizes(n_leaves: int) -> List[int]:
    sizes, cur = [], n_leaves
    while cur > 1:
        cur //= 2
        sizes.append(cur)
    return sizes


class _SpanLevels(torch.autograd.Function):
    """The level loop of `HierarchicalAttention.cross_update_Y` (reference
    hierarchical_attention/modules/attention.py:101-157, everything before out_proj_y) as one
    differentiable function on fused projections.  The reference gets the same gradients from
    autograd through 3 + 2L Linear layers and L `BuildParentNodesFunc`s (ops/functional.py:66-111)."""

    @staticmethod
    def forward(ctx, module, drop_p, x, y_in, wq, wk, wv):
        y_new, kept = module._span_levels(x, y_in, keep=True, drop_p=drop_p)
        # everything the backward reads goes through save_for_backward: an in-place write to one
        # of these tensors between forward and backward is then reported by autograd instead of
        # giving wrong gradients, and saved-tensor hooks (checkpointing, offloading) see them
        nl = len(kept["kvs"])
        ctx.save_for_backward(kept["x"], kept["y_in"], kept["qkv"], kept["blocks"], kept["w_qkv"], kept["w_kv"],
                              *kept["kvs"], *kept["masks"], *kept["chain"])
        ctx.module, ctx.levels, ctx.scales, ctx.masks = module, nl, kept["scales"], len(kept["masks"])
        ctx.in_dtypes = (x.dtype, y_in.dtype, wq.dtype)
        return y_new

    @staticmethod
    def backward(ctx, dy):
        # raises autograd's own error if they were freed or modified; saved-tensor hooks may give back
        # another layout, the kernels read them as dense
        saved = [t.contiguous() for t in ctx.saved_tensors]
        nl = ctx.levels
        kept = dict(zip(("x", "y_in", "qkv", "blocks", "w_qkv", "w_kv"), saved[:6]))
        kept["kvs"], kept["masks"], kept["scales"] = list(saved[6:6 + nl]), list(saved[6 + nl:6 + nl + ctx.masks]), ctx.scales
        kept["chain"] = saved[6 + nl + ctx.masks:]
        dx, dy_in, dw = ctx.module._span_levels_backward(dy, kept)
        xd, yd, wd = ctx.in_dtypes
        D = dx.shape[-1]
        dw = dw.to(wd)
        return None, None, dx.to(xd), dy_in.to(yd), dw[:D], dw[D:2 * D], dw[2 * D:]


class HierarchicalAttention(nn.Module):
    def __init__(self, dim: int, num_heads: int, dropout: float = 0.1, window_size: int = 16):
        super().__init__()
        assert dim % num_heads == 0, "dim must be divisible by num_heads"
        self.dim, self.num_heads, self.head_dim = dim, num_heads, dim // num_heads
        self.window_size = window_size
        # bottom-up (span nodes)
        self.Wq_y = nn.Linear(dim, dim, bias=False)
        self.Wk_y = nn.Linear(dim, dim, bias=False)
        self.Wv_y = nn.Linear(dim, dim, bias=False)
        self.out_proj_y = nn.Linear(dim, dim)
        # top-down (leaves)
        self.Wq_x = nn.Linear(dim, dim, bias=False)
        self.Wk_x = nn.Linear(dim, dim, bias=False)
        self.Wv_x = nn.Linear(dim, dim, bias=False)
        self.out_proj_x = nn.Linear(dim, dim)
        self.dropout = nn.Dropout(dropout)
        # topology cache: one set of tables per (length, causal, device)
        self.cached_tables = None
        self.cached_seq_len = -1
        self.cached_is_causal = None
        self.sizes: Optional[List[int]] = None
        self.offsets: Optional[List[int]] = None
        self._fused = {}  # row-concatenated projection weights of the no-autograd path
        self.fuse_top_levels = True  # no-autograd path: the last levels in one launch where the shape allows
        self.fused_training = True   # autograd path: fused projections and one backward kernel per level

    # -- helpers -------------------------------------------------------------
    def _get_lookup_table(self, L: int, is_causal: bool, device: torch.device):
        t = self.cached_tables
        if (t is None or self.cached_seq_len != L or self.cached_is_causal != is_causal
                or t["forward_idx"].device != device):
            t = build_tree_topology(L, is_causal=is_causal, device=device)
            self.cached_tables, self.cached_seq_len, self.cached_is_causal = t, L, is_causal
        return t

    def _build_level_info(self, N: int):
        sizes = _level_sizes(N)
        offsets = [0]
        for s in sizes[:-1]:
            offsets.append(offsets[-1] + s)
        return sizes, offsets

    # update_X_from_Y without autograd where the projections do not go into one launch: keys and values straight into
    # their rows from this many 16-bit elements of x on, or half as many 32-bit ones (us for the whole call, so /
    # from the joined input, 1024 channels unless said: bf16 B2 N1024 159 / 109, B4 N2048 163 / 138, B8 N2048 242 / 236, B8
    # N4096 470 / 477; fp16 146 / 109, 151 / 142, 220 / 246, 416 / 495; bf16 autocast 189 / 133, 214 / 201, 337 / 365, 625 /
    # 713; fp32 B1 N2048 of 512 150 / 115, B8 N1024 of 640 391 / 386, B4 N2048 789 / 809, B8 N4096 3113 / 3205)
    _DIRECT_PROJECTION_MIN_ELEMENTS = 1 << 24
    # training: levels of at most this many children over the batch run as fused chains, forward and backward
    # (no chain / 1024 / 4096, us forward and backward of one module, fp16: B8 N2048 d768 2034 / 1996 / 1967, B2
    # N512 d512 1503 / 1096 / 1102, B4 N64 d768 1330 / 1084 / 1089, B1 N4096 d1024 1649 / 1232 / 1159)
    _TRAINING_CHAIN_ROWS = 4096

    def _heads(self, t: torch.Tensor) -> torch.Tensor:
        return t.view(t.shape[0], -1, self.num_heads, self.head_dim)

    def reset_fused_weights(self):
        """Drops the cached stacked / packed projection weights of the no-autograd path.  The cache
        notices optimizer steps, `load_state_dict`, `.to()` and `train()` by itself; call this after
        writing to a weight through `.data` (such writes leave no trace on the tensor)."""
        self._fused.clear()

    def _load_from_state_dict(self, *args, **kwargs):
        self._fused.clear()
        return super()._load_from_state_dict(*args, **kwargs)

    def _apply(self, fn, *args, **kwargs):
        self._fused.clear()
        return super()._apply(fn, *args, **kwargs)

    def train(self, mode: bool = True):
        self._fused.clear()
        return super().train(mode)

    def _fused_weight(self, name: str, layers, dtype: torch.dtype, packed: bool = False) -> torch.Tensor:
        """Weights of several bias-free projections, cast to `dtype` and stacked along the output
        dimension, so one GEMM computes them all (packed: key / value weights in the operand order
        of the fused upper levels); rebuilt when any of them has been written to or moved."""
        params = [weight_and_bias(m)[0] for m in layers]
        key = tuple((w.data_ptr(), w._version, w.dtype) for w in params) + (dtype,)
        hit = self._fused.get(name)
        if hit is None or hit[0] != key:
            ws = [w.detach().to(dtype) for w in params]
            hit = (key, pack_kv_weights(ws[0], ws[1], self.num_heads) if packed else torch.cat(ws, dim=0))
            # (under capture the copy holds nothing before the first replay: it stays with the graph)
            if not (params[0].is_cuda and torch.cuda.is_current_stream_capturing()):
                self._fused[name] = hit
        return hit[1]

    def _chain_weights(self, x: torch.Tensor):
        """(q | k | v, packed k / v) weights of the span nodes' update of leaves x as one chain of fused levels in
        x's type, or None where that does not apply."""
        if x.dtype not in (torch.float16, torch.bfloat16) or x.dim() != 3:
            return None
        layers = [self._modules[n] for n in ("Wq_y", "Wk_y", "Wv_y")]
        if any(m._parameters["weight"].dtype != x.dtype or m._parameters["weight"].device != x.device for m in layers):
            return None
        if _lib.lib().hsa_cross_update_level_rows(x.shape[0], self.num_heads, self.head_dim, _lib.dtype_code(x)) < x.shape[1]:
            return None
        with _lib.on_device(x):
            return (self._fused_weight("qkv_y", layers, x.dtype),
                    self._fused_weight("kv_y_packed", layers[1:], x.dtype, packed=True))

    @staticmethod
    def _compute_dtype(t: torch.Tensor) -> torch.dtype:
        """Element type the projections produce: the autocast type inside `torch.autocast` (the
        reference's evaluation loop runs under it with fp32 activations and weights), else the
        activations' own type."""
        if t.is_cuda and torch.is_autocast_enabled("cuda"):
            return torch.get_autocast_dtype("cuda")
        return t.dtype

    def _needs_autograd(self, tensors, layers) -> bool:
        if not torch.is_grad_enabled():
            return False
        return any(t.requires_grad for t in tensors) or any(
            p.requires_grad for m in layers for p in m.parameters())

    def _span_levels(self, x: torch.Tensor, y_in: torch.Tensor, keep: bool = False, drop_p: float = 0.0):
        """The level loop of cross_update_Y on fused projections, without autograd: the three
        projections of the span nodes are one GEMM, the key/value projections of each level's
        children another, and each level's kernel reads its operands as column slices of those
        results.  Every level writes twice: a dense [B, P, D] block that feeds the next level's
        GEMM, and its slice of the level-concatenated [B, N-1, D] result (returned, before
        out_proj_y).  Unless `keep`, the last levels (few rows each) run as one launch that does
        their projections on chip.  `keep` returns what a backward pass needs as a dict; `drop_p`
        is the dropout probability applied to the children's values (the reference applies it
        twice to the leaves' values)."""
        B, N, D = x.shape
        H, Dh = self.num_heads, self.head_dim
        _lib.require_gpu(x, y_in)
        cdt = self._compute_dtype(x)
        x, y_in = x.to(cdt).contiguous(), y_in.to(cdt).contiguous()
        w_qkv = self._fused_weight("qkv_y", (self.Wq_y, self.Wk_y, self.Wv_y), cdt)
        qkv = project(y_in, w_qkv)  # [B, N-1, 3D]
        w_kv = self._fused_weight("kv_y", (self.Wk_y, self.Wv_y), cdt)
        # every buffer the kernels address by raw pointer has the one element type
        assert qkv.dtype == cdt and qkv.is_contiguous(), "projection result has an unexpected layout"
        y_new = torch.empty((B, N - 1, D), dtype=cdt, device=x.device)
        blocks = torch.empty(B * (N - 1) * D, dtype=cdt, device=x.device)  # level-major
        # the level loop works on raw addresses: the operands are fixed column slices of qkv and
        # of each level's k/v projection, so no tensor views are made per level
        es = x.element_size()
        A = ctypes.c_int64 * 7
        row_strides = A(3 * D, 3 * D, 3 * D, 2 * D, 2 * D, D, D)
        fwd, code, stream = _lib.lib().hsa_build_parents_strided_fwd, _lib.dtype_code(x), _lib.stream_of(x)
        qkv_p, blk_p, out_p = qkv.data_ptr(), blocks.data_ptr(), y_new.data_ptr()
        # child rows the fused upper levels take (0: shape not handled)
        # (y_new's rows are 16-byte aligned: the fused upper levels may run as a launch per level)
        top_rows = 0
        # (training at widths of an odd number of 64 channels: the levels by themselves are as fast, B4 N2048 d832 1369
        # / 1369, or faster, B8 N128 d448 935 / 970 us forward and backward)
        if self.fuse_top_levels and not (keep and (drop_p > 0 or D % 128)):
            top_rows = _lib.lib().hsa_cross_update_level_rows(B, H, Dh, code)
            if keep:  # (the projected rows are needed again: only where launches are what counts)
                top_rows = min(top_rows, self._TRAINING_CHAIN_ROWS // B)
        kvs, masks, scales, chain = [], [], [], ()
        src, off = x, 0
        with _lib.on_device(x):
            for lvl, P in enumerate(self.sizes):
                if 2 * P <= top_rows:
                    # the remaining levels: fused projection + parent build, no GEMM launches
                    w_top = self._fused_weight("kv_y_packed", (self.Wk_y, self.Wv_y), cdt, packed=True)
                    assert src.dtype == cdt and src.is_contiguous() and w_top.dtype == cdt
                    rc = _lib.lib().hsa_cross_update_top_fwd(
                        src.data_ptr(), qkv_p + off * 3 * D * es, w_top.data_ptr(), out_p + off * D * es,
                        B, 2 * P, H, Dh, 0, (N - 1) * 3 * D, 3 * D, (N - 1) * D, D, code, stream)
                    _lib.check(rc, "hsa_cross_update_top_fwd")
                    if keep:
                        # the backward's keys and values of these levels' children, one GEMM for all
                        rows = torch.cat([src, y_new[:, off:N - 2]], dim=1)  # [B, 4P-2, D]
                        chain = (rows, project(rows, w_kv))
                    break
                kv = project(src, w_kv)  # [B, 2P, 2D]
                assert kv.dtype == cdt and kv.is_contiguous(), "projection result has an unexpected layout"
                if drop_p > 0:
                    # dropout on the value half: a saved boolean keep-mask (drawn in fp32) and one
                    # scale applied as a scalar, i.e. in fp32 with a single rounding of the product
                    # (a mask holding 1/keep_p in bf16 would scale by 1.109 instead of 1.111)
                    keep_p = 1.0 - drop_p
                    m = torch.rand((B, 2 * P, D), dtype=torch.float32, device=x.device) < keep_p
                    scale = 1.0 / keep_p
                    if lvl == 0:  # the leaves' values pass through dropout twice
                        m &= torch.rand((B, 2 * P, D), dtype=torch.float32, device=x.device) < keep_p
                        scale = scale * scale
                    kv[:, :, D:].mul_(m).mul_(scale)
                    masks.append(m)
                    scales.append(scale)
                par, kv_p, lvl_p = qkv_p + off * 3 * D * es, kv.data_ptr(), blk_p + B * off * D * es
                rc = fwd(par, par + D * es, par + 2 * D * es, kv_p, kv_p + D * es, lvl_p,
                         out_p + off * D * es, B, P, H, Dh,
                         A((N - 1) * 3 * D, (N - 1) * 3 * D, (N - 1) * 3 * D, 4 * P * D, 4 * P * D, P * D,
                           (N - 1) * D), row_strides, code, stream)
                _lib.check(rc, "hsa_build_parents_strided_fwd")
                if keep:
                    kvs.append(kv)
                src = blocks[B * off * D:B * (off + P) * D].view(B, P, D)
                off += P
        if not keep:
            return y_new
        return y_new, {"x": x, "y_in": y_in, "qkv": qkv, "blocks": blocks, "kvs": kvs, "masks": masks,
                       "scales": scales, "w_qkv": w_qkv, "w_kv": w_kv, "chain": chain}

    def _span_levels_backward(self, dy: torch.Tensor, kept: dict):
        """Gradients of `_span_levels` with respect to x, y_in and the stacked q|k|v weights:
        per level one kernel (the three weights are recomputed, every gradient row written once
        into the fused layouts) and one GEMM (gradient of the level's input); the weight gradients
        of all levels are one contraction at the end.  The last levels, where the forward ran them as
        a chain, are one launch each.  Returns (dx, dy_in, dW_qkv [3D, D])."""
        x, y_in, qkv, blocks = kept["x"], kept["y_in"], kept["qkv"], kept["blocks"]
        kvs, masks, w_qkv, w_kv = kept["kvs"], kept["masks"], kept["w_qkv"], kept["w_kv"]
        B, N, D = x.shape
        H, Dh = self.num_heads, self.head_dim
        cdt, es = x.dtype, x.element_size()
        sizes, offsets = self._build_level_info(N)
        dy = dy.to(cdt).contiguous()
        if dy.data_ptr() % 16:  # the chain's kernels move row pieces
            dy = dy.clone()
        dqkv = torch.empty_like(qkv)
        # level-major like `blocks`: the children of level 1 (the leaves), then those of the levels above
        inner = B * offsets[len(kvs) - 1] if kvs else 0  # rows of all children above the leaves
        dkv = torch.empty((B * N + inner if kvs else 0, 2 * D), dtype=cdt, device=x.device)
        A = ctypes.c_int64 * 11
        bwd, code, stream = _lib.lib().hsa_build_parents_level_bwd, _lib.dtype_code(x), _lib.stream_of(x)
        rs = A(D, 3 * D, 3 * D, 3 * D, 2 * D, 2 * D, 3 * D, 3 * D, 3 * D, 2 * D, 2 * D)
        T3 = (N - 1) * 3 * D
        d_above = None
        pairs = [(dqkv.view(-1, 3 * D), y_in.view(-1, D), 0)]
        with _lib.on_device(x):
            if kept["chain"]:
                rows, kv = kept["chain"]
                dkv_up, C, off = torch.empty_like(kv), 2 * sizes[len(kvs)], offsets[len(kvs)]
                # the weights in the order the kernel multiplies them: [head][16-column tile][step][4][16][8]
                w_ops = w_kv.view(2 * D // 32, 4, 8, H, Dh // 16, 16).permute(3, 4, 0, 1, 5, 2).contiguous()
                rc = _lib.lib().hsa_span_levels_bwd(
                    dy.data_ptr() + off * D * es, qkv.data_ptr() + off * 3 * D * es, kv.data_ptr(), w_ops.data_ptr(),
                    dqkv.data_ptr() + off * 3 * D * es, dkv_up.data_ptr(), B, C, H, Dh, (N - 1) * D, D, T3, 3 * D, T3,
                    3 * D, code, stream)
                _lib.check(rc, "hsa_span_levels_bwd")
                d_above = project(dkv_up[:, :C].reshape(-1, 2 * D), w_kv, True)  # [B * C, D]
                pairs.append((dkv_up.view(-1, 2 * D), rows.view(-1, D), D))
            for lvl in range(len(kvs) - 1, -1, -1):
                P, off = sizes[lvl], offsets[lvl]
                kv = kvs[lvl]
                row = 0 if lvl == 0 else B * (N + offsets[lvl - 1])
                dkv_l = dkv[row:row + 2 * B * P]
                par, dpar = qkv.data_ptr() + off * 3 * D * es, dqkv.data_ptr() + off * 3 * D * es
                kv_p, dkv_p = kv.data_ptr(), dkv_l.data_ptr()
                rc = bwd(dy.data_ptr() + off * D * es, None if d_above is None else d_above.data_ptr(),
                         par, par + D * es, par + 2 * D * es, kv_p, kv_p + D * es,
                         dpar, dpar + D * es, dpar + 2 * D * es, dkv_p, dkv_p + D * es, B, P, H, Dh,
                         A((N - 1) * D, T3, T3, T3, 4 * P * D, 4 * P * D, T3, T3, T3, 4 * P * D, 4 * P * D), rs, code,
                         stream)
                _lib.check(rc, "hsa_build_parents_level_bwd")
                if masks:
                    dkv_l.view(B, 2 * P, 2 * D)[:, :, D:].mul_(masks[lvl]).mul_(kept["scales"][lvl])
                d_above = project(dkv_l, w_kv, True)  # [B * 2P, D]
        dx = d_above.view(B, N, D)
        dy_in = project(dqkv, w_qkv, True)
        if kvs:
            pairs.append((dkv[:B * N], x.view(-1, D), D))
        if inner:
            pairs.append((dkv[B * N:], blocks[:inner * D].view(inner, D), D))
        res = _lib.ext().weight_grad(pairs, 3 * D, torch.float32, False)
        if res is not None:
            return dx, dy_in, res[0]
        dw_qkv = torch.matmul(pairs[0][0].t(), pairs[0][1]).float()
        for g, src, _ in pairs[1:]:
            dw_qkv[D:] += torch.matmul(g.t(), src).float()
        return dx, dy_in, dw_qkv

    # -- bottom-up: leaves -> span nodes ----------------------------------------
    def cross_update_Y(self, x: torch.Tensor, y_in: torch.Tensor) -> torch.Tensor:
        B, N, D = x.shape
        assert y_in is not None, "y_in cannot be None"
        assert y_in.size(1) == N - 1, \
            f"y_in size {y_in.size(1)} mismatch! Expected N-1 ({N-1}) for N={N} leaves."
        if self.sizes is None or self.sizes[0] != N // 2:
            self.sizes, self.offsets = self._build_level_info(N)

        grad = self._needs_autograd((x, y_in), (self.Wq_y, self.Wk_y, self.Wv_y))
        drop_p = self.dropout.p if self.training else 0.0
        if not grad and drop_p == 0:
            return linear(self.out_proj_y, self._span_levels(x, y_in))
        if self.fused_training and x.is_cuda and N >= 2:
            # the same fused level loop as one differentiable function
            y_new = _SpanLevels.apply(self, drop_p, x, y_in, self.Wq_y.weight, self.Wk_y.weight, self.Wv_y.weight)
            return linear(self.out_proj_y, y_new)

        q_lv = torch.split(self._heads(self.Wq_y(y_in)), self.sizes, dim=1)
        k_lv = torch.split(self._heads(self.Wk_y(y_in)), self.sizes, dim=1)
        v_lv = torch.split(self._heads(self.Wv_y(y_in)), self.sizes, dim=1)
        levels, src = [], x
        for lvl, P in enumerate(self.sizes):
            k_c = self._heads(self.Wk_y(src))
            v_c = self.dropout(self._heads(self.Wv_y(src)))
            if lvl == 0:
                v_c = self.dropout(v_c)  # the leaf values pass through dropout twice
            src = build_parent_nodes(q_lv[lvl], k_lv[lvl], v_lv[lvl], k_c, v_c).reshape(B, P, D)
            levels.append(src)
        return self.out_proj_y(torch.cat(levels, dim=1))

    # -- top-down: span nodes -> leaves -------------------------------------------
    def update_X_from_Y(self, x: torch.Tensor, y: torch.Tensor,
                        mask: Optional[torch.Tensor] = None) -> torch.Tensor:
        B, N, D = x.shape
        assert y is not None, "y (parents) cannot be None during top-down update"
        grad = self._needs_autograd((x, y), (self.Wq_x, self.Wk_x, self.Wv_x))
        dropped = self.training and self.dropout.p > 0
        join = query_key_value_rows if grad else query_key_value
        qkv = join(self.Wq_x, self.Wk_x, self.Wv_x, x, y)
        q = self._heads(linear(self.Wq_x, x) if qkv is None else qkv[0])
        if (qkv is None and not grad and not dropped and y.size(1) == N - 1
                and B * N * D * q.element_size() >= 2 * self._DIRECT_PROJECTION_MIN_ELEMENTS):
            # leaves and span nodes are projected straight into their rows of the [B, 2N-1, D]
            # key / value buffers (batched GEMMs with a strided output): no concatenated input.
            # (Four batched GEMM launches instead of a copy and two plain ones: all but large inputs, where the
            # launches cost more host time than the copy costs the GPU, take the other branch.)
            # Everything is brought to the type of q first (under autocast the activations and
            # weights are fp32 while the projections come out in the autocast type; GEMMs with an
            # `out=` are not autocast)
            cdt = q.dtype
            xc, yc = x.to(cdt), y.to(cdt)
            k = torch.empty((B, 2 * N - 1, D), dtype=cdt, device=x.device)
            v = torch.empty_like(k)
            # (bf16: weights laid out along the contraction, since torch's batched bf16 product of a transposed right
            # operand has faulted on this device: 7 us for each of 1024 x 1024, at every call, since a kept copy would miss
            # writes through .data and in a graph any write; fp16: as they are, 8 x 2048 x 1024 x 1024 33 us against 40)
            for lin, dst in ((self.Wk_x, k), (self.Wv_x, v)):
                wt = lin.weight.detach().to(cdt).t()
                wt = (wt.contiguous() if cdt == torch.bfloat16 else wt).unsqueeze(0).expand(B, D, D)
                torch.bmm(xc, wt, out=dst[:, :N])
                torch.bmm(yc, wt, out=dst[:, N:])
            k, v = self._heads(k), self._heads(v)
        else:
            if qkv is None:
                xy = torch.cat([x, y], dim=1)
                k, v = linear(self.Wk_x, xy), linear(self.Wv_x, xy)
            else:
                k, v = qkv[1:]
            k, v = self._heads(k), self.dropout(self._heads(v))
        is_causal = mask is not None  # only the presence of a mask is looked at
        t = self._get_lookup_table(N, is_causal, x.device)
        heads = hierarchical_attention(q, k, v, t["forward_idx"], t["backward_gather"],
                                       t["forward_mask"] if is_causal else None, self.window_size)
        return linear(self.out_proj_x, heads.view(B, N, D))

    def _batched(self, a: torch.Tensor, b: torch.Tensor) -> torch.Tensor:
        """a @ b over the leading dimensions.  bf16 on the GPU: the same operands in fp32, one rounding, also in
        the backward (torch's batched bf16 product of a transposed right operand has faulted on this device, and
        the backward of any makes such a product)."""
        dtype = self._compute_dtype(a)
        if not a.is_cuda or dtype != torch.bfloat16:
            return torch.matmul(a, b)
        with torch.autocast("cuda", enabled=False):
            return torch.matmul(a.to(dtype).float(), b.to(dtype).float()).to(dtype)

    def _standard_attention(self, Q, K, V, mask):
        scores = self._batched(Q, K.transpose(-1, -2)) / math.sqrt(Q.size(-1))
        if mask is not None:
            scores = scores.masked_fill(mask == 0, float("-inf"))
        attn = self.dropout(torch.softmax(scores, dim=-1))
        return self._batched(attn, V), attn

    def forward(self, query, key, value, y=None, mask=None, return_attention=False):
        B, Lq, D = query.shape
        if y is not None and Lq == key.size(1) == value.size(1):
            out = self.update_X_from_Y(query, y, mask)
            return (out, None) if return_attention else out
        # dense fallback when no span nodes are given or the lengths differ
        H, Dh = self.num_heads, self.head_dim
        Q = self.Wq_x(query).view(B, Lq, H, Dh).transpose(1, 2)
        K = self.Wk_x(key).view(B, key.size(1), H, Dh).transpose(1, 2)
        V = self.Wv_x(value).view(B, value.size(1), H, Dh).transpose(1, 2)
        ctx, attn = self._standard_attention(Q, K, V, mask)
        out = self.out_proj_x(ctx.transpose(1, 2).reshape(B, Lq, D))
        return (out, attn) if return_attention else out


FORWARDS[HierarchicalAttention] = HierarchicalAttention.forward
