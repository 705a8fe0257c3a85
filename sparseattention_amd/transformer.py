"""Decoder-only language model built on `HierarchicalAttention`: the caller of the hot path.

Restates the model of the reference's training script
(hierarchical_attention_project/Hierarchical_Transformer_Pretrain.py:331-481) with the same
sub-module names, so its checkpoints (`model_state_dict`, optionally with a `module.` prefix)
load unchanged.  Differences: the feed-forward activation is selectable (the reference uses
ReLU), and the causal "mask" handed to the attention is a one-element tensor, because only its
presence is ever looked at (an N x N mask costs 16 MB at N=4096 and is never read).
"""
from __future__ import annotations

import math
import operator
import sys

import torch
import torch.nn as nn
import torch.nn.functional as F

from . import _lib
from .modules import HierarchicalAttention
from .modules import attention as _attention
from .ops import generate_span_input_Y
from .ops.linear import FORWARDS, all_plain, linear, plain_module, watched, weight_and_bias


def _norm_weights(m):
    """Weight and bias of an nn.LayerNorm over the last dimension with both that may be bypassed, else None."""
    if not plain_module(m, nn.LayerNorm) or len(m.normalized_shape) != 1:
        return None
    w, b = weight_and_bias(m)
    return None if w is None or b is None else (w, b)


def layer_norm(x, norm):
    """norm(x) on this package's kernel where it takes the case."""
    wb = _norm_weights(norm) if x.is_cuda and not torch.is_autocast_enabled("cuda") else None
    if wb is not None and not watched(x, *wb):
        r = _lib.ext().add_layer_norm(x, None, *wb, norm.eps)
        if r is not None:
            return r[1]
    return norm(x)


def add_layer_norm(x, branch, norm):
    """(x + branch, norm(x + branch)): one kernel reads both once and writes both results, where it
    takes the case (one GPU, one element type; autocast mixes types and keeps the two steps)."""
    wb = _norm_weights(norm) if x.is_cuda and not torch.is_autocast_enabled("cuda") else None
    if wb is not None and not watched(x, branch, *wb):
        r = _lib.ext().add_layer_norm(x, branch, *wb, norm.eps)
        if r is not None:
            return r
    x = x + branch
    return x, norm(x)


class PositionwiseFeedForward(nn.Module):
    def __init__(self, d_model: int, d_ff: int, dropout: float = 0.1, activation: str = "relu"):
        super().__init__()
        self.fc1 = nn.Linear(d_model, d_ff)
        self.fc2 = nn.Linear(d_ff, d_model)
        self.dropout = nn.Dropout(p=dropout)
        self.activation = {"relu": F.relu, "gelu": F.gelu}[activation]

    def forward(self, x):
        return linear(self.fc2, self.dropout(self.activation(linear(self.fc1, x))))


FORWARDS[PositionwiseFeedForward] = PositionwiseFeedForward.forward


class PositionalEncoding(nn.Module):
    def __init__(self, d_model: int, dropout: float, max_len: int = 5000):
        super().__init__()
        self.dropout = nn.Dropout(p=dropout)
        pos = torch.arange(0.0, max_len).unsqueeze(1)
        freq = torch.exp(torch.arange(0.0, d_model, 2) * -(math.log(10000.0) / d_model))
        pe = torch.zeros(max_len, d_model)
        pe[:, 0::2] = torch.sin(pos * freq)
        pe[:, 1::2] = torch.cos(pos * freq)
        self.register_buffer("pe", pe.unsqueeze(0))

    def forward(self, x):
        return self.dropout(x + self.pe[:, :x.size(1), :].to(x.dtype))


class DecoderLayer(nn.Module):
    def __init__(self, d_model, num_heads, d_ff, dropout=0.1, window_size=16, activation="relu"):
        super().__init__()
        self.self_attn = HierarchicalAttention(d_model, num_heads, dropout, window_size=window_size)
        self.feed_forward = PositionwiseFeedForward(d_model, d_ff, dropout, activation)
        self.norm1 = nn.LayerNorm(d_model)
        self.norm2 = nn.LayerNorm(d_model)
        self.norm_y = nn.LayerNorm(d_model)
        # present in the reference's checkpoints, unused by its forward
        self.alpha_proj = nn.Linear(d_model, d_model)
        self.beta_proj = nn.Linear(d_model, d_model)
        self.dropout = nn.Dropout(dropout)

    def forward(self, x, y, mask=None, return_attention=False):
        if return_attention:
            # span nodes first: un-normalised leaves, normalised nodes; plain residual
            y = y + self.dropout(self.self_attn.cross_update_Y(x, y_in=self.norm_y(y)))
            # leaves: pre-norm attention over the window and the updated nodes
            nx = self.norm1(x)
            a, w = self.self_attn(nx, nx, nx, y=y, mask=mask, return_attention=True)
            x = x + self.dropout(a)
            x = x + self.dropout(self.feed_forward(self.norm2(x)))
            return x, y, w
        return self._chained(x, y, layer_norm(x, self.norm1), layer_norm(y, self.norm_y), mask)[:2]

    def _chained(self, x, y, nx, ny, mask, following=None):
        """The layer on inputs whose norms are there already (nx = norm1(x), ny = norm_y(y)).  With
        `following`, the layer that comes next, its norms of the results are taken together with the
        residual sums and returned as well: (x, y, nx, ny)."""
        u = self.dropout(self.self_attn.cross_update_Y(x, y_in=ny))
        y, ny = (y + u, None) if following is None else add_layer_norm(y, u, following.norm_y)
        a = self.self_attn(nx, nx, nx, y=y, mask=mask)
        x, n2 = add_layer_norm(x, self.dropout(a), self.norm2)
        f = self.dropout(self.feed_forward(n2))
        x, nx = (x + f, None) if following is None else add_layer_norm(x, f, following.norm1)
        return x, y, nx, ny

    def _native(self, x, y, nx, ny, mask, following=None):
        """`_chained` without autograd as one native call (csrc/torch_ops.cpp), launch for launch the same; None
        where something may watch or replace one of its steps, or where the call does not take the layer."""
        if torch.is_grad_enabled() or not x.is_cuda or torch.compiler.is_compiling() or watched(x, y, nx, ny):
            return None
        sub = self._modules
        att, ff = sub["self_attn"], sub["feed_forward"]
        if type(att) is not HierarchicalAttention or type(ff) is not PositionwiseFeedForward:
            return None
        a, f = att._modules, ff._modules
        wq = a["Wq_x"]._parameters.get("weight")
        if wq is None or not _lib.ext().decoder_layer_takes(x, y, wq, att.num_heads):
            return None
        # (written for its host time, which a short sequence waits for: sets of types and plain loops)
        drops = [sub["dropout"], a["dropout"], f["dropout"]]
        norms = [sub["norm2"]]
        if following is not None:
            norms += [following._modules["norm_y"], following._modules["norm1"]]
        linears = [a["out_proj_y"], a["Wq_x"], a["Wk_x"], a["Wv_x"], a["out_proj_x"], f["fc1"], f["fc2"]]
        if not all_plain([(att, HierarchicalAttention), (ff, PositionwiseFeedForward), *zip(drops, _DROPS), *zip(norms, _NORMS),
                          *zip(linears, _LINEARS)]):
            return None
        for m in drops:
            if m.training and m.p > 0:
                return None
        for m in norms:
            if len(m.normalized_shape) != 1:
                return None
        if not att.fuse_top_levels or not _own_steps(self, att) or (ff.activation is not F.gelu and ff.activation is not F.relu):
            return None
        # (weights and norms: parameters, neither missing nor plain tensors in their places; their type and sizes are
        # the native call's to check)
        linears = [m._parameters for m in linears]
        w, b = [p.get("weight") for p in linears], [p.get("bias") for p in linears]
        n = []
        for m in norms:
            m = m._parameters
            n += m.get("weight"), m.get("bias")
        spans = [a["Wq_y"]._parameters.get("weight"), a["Wk_y"]._parameters.get("weight"), a["Wv_y"]._parameters.get("weight")]
        if {*map(type, w), *map(type, n), *map(type, spans)} != _PARAMETERS:
            return None
        if (b[0] is None or b[1] is not None or b[2] is not None or b[3] is not None or b[4] is None or b[5] is None
                or b[6] is None):
            return None
        packed = att._chain_weights(x)
        if packed is None:
            return None
        params = [*packed, w[0], b[0], w[1], w[2], w[3], w[4], b[4], n[0], n[1], w[5], b[5], w[6], b[6], *n[2:]]
        eps = [m.eps for m in norms] + [0.0] * (3 - len(norms))
        return _lib.ext().decoder_layer(x, y, nx, ny, params, eps, att.num_heads, att.window_size, mask is not None,
                                        ff.activation is F.gelu, following is not None)

    def _may_chain(self) -> bool:
        """Whether `_chained` may stand in for calling the layer."""
        return plain_module(self, DecoderLayer)


FORWARDS[DecoderLayer] = DecoderLayer.forward
# what the native layer stands in for besides its modules' forwards, as it is when this module is loaded
_STEPS = tuple((owner, name, getattr(owner, name)) for owner, names in (
    (HierarchicalAttention, ("cross_update_Y", "update_X_from_Y", "_span_levels", "_fused_weight", "_chain_weights")),
    (DecoderLayer, ("_chained",)),
    (_attention, ("hierarchical_attention", "linear", "project", "query_key_value")),
    (sys.modules[__name__], ("add_layer_norm", "linear"))) for name in names)


_STEP_OWNERS, _STEP_NAMES, _STEP_FUNCTIONS = zip(*_STEPS)
_ATTENTION_STEPS = [name for owner, name, _ in _STEPS if owner is HierarchicalAttention]
_DROPS, _NORMS, _LINEARS, _PARAMETERS = (nn.Dropout,) * 3, (nn.LayerNorm,) * 3, (nn.Linear,) * 7, {nn.Parameter}


def _own_steps(layer, att) -> bool:
    """Nobody has replaced one of the steps, on its class, on the instance or in its module."""
    return (all(map(operator.is_, map(getattr, _STEP_OWNERS, _STEP_NAMES), _STEP_FUNCTIONS))
            and "_chained" not in layer.__dict__ and att.__dict__.keys().isdisjoint(_ATTENTION_STEPS))


class TransformerLM(nn.Module):
    def __init__(self, vocab_size, d_model, num_heads, d_ff, num_layers, dropout=0.1, window_size=16,
                 activation="relu", max_len=5000):
        super().__init__()
        self.embedding = nn.Embedding(vocab_size, d_model)
        self.pos_encoding = PositionalEncoding(d_model, dropout=dropout, max_len=max_len)
        self.layers = nn.ModuleList(
            [DecoderLayer(d_model, num_heads, d_ff, dropout, window_size, activation) for _ in range(num_layers)])
        self.fc_out = nn.Linear(d_model, vocab_size)
        self.fc_out.weight = self.embedding.weight  # tied
        self.d_model = d_model
        self.apply(self._init_weights)

    @staticmethod
    def _init_weights(m):
        if isinstance(m, nn.Linear):
            nn.init.normal_(m.weight, mean=0.0, std=0.02)
            if m.bias is not None:
                nn.init.zeros_(m.bias)
        elif isinstance(m, nn.Embedding):
            nn.init.normal_(m.weight, mean=0.0, std=0.02)

    def make_causal_mask(self, x):
        """Only `mask is not None` is ever tested downstream."""
        return torch.ones(1, 1, 1, 1, dtype=torch.bool, device=x.device)

    def forward(self, trg, return_attention=False):
        x = self.pos_encoding(self.embedding(trg) * math.sqrt(self.d_model))
        y = generate_span_input_Y(x)
        mask = self.make_causal_mask(trg)
        layers = list(self.layers)
        if layers and not return_attention and all(type(m) is DecoderLayer and m._may_chain() for m in layers):
            nx, ny = layer_norm(x, layers[0].norm1), layer_norm(y, layers[0].norm_y)
            for layer, following in zip(layers, layers[1:] + [None]):
                done = layer._native(x, y, nx, ny, mask, following)
                x, y, nx, ny = layer._chained(x, y, nx, ny, mask, following) if done is None else done
            return linear(self.fc_out, x, wide=True)
        for layer in layers:
            if return_attention:
                x, y, _ = layer(x, y, mask=mask, return_attention=True)
            else:
                x, y = layer(x, y, mask=mask)
        return self.fc_out(x)

    def generate(self, src, start_token=2, max_len=50, temperature=1.0):
        """Samples up to `max_len` tokens after the prompt `src`, one full forward per token, and
        stops at the end-of-sequence id 3 (Hierarchical_Transformer_Pretrain.py:483-505).  As in the
        reference every forward needs a power-of-two length, so only prompts whose length stays a
        power of two while tokens are appended get past the first step."""
        self.eval()
        device = next(self.parameters()).device
        tokens = src.to(device)
        if tokens.dim() == 1:
            tokens = tokens.unsqueeze(0)
        with torch.no_grad():
            for _ in range(max_len):
                logits = self.forward(tokens)
                probs = torch.softmax(logits[:, -1, :] / temperature, dim=-1)
                nxt = torch.multinomial(probs, 1)
                tokens = torch.cat([tokens, nxt], dim=1)
                if nxt.item() == 3:
                    break
        return tokens

    def load_reference_checkpoint(self, state):
        """Loads a reference checkpoint dict (`{'model_state_dict': ...}` or a bare state dict,
        keys optionally prefixed with `module.`)."""
        sd = state.get("model_state_dict", state)
        sd = {(k[7:] if k.startswith("module.") else k): v for k, v in sd.items()}
        return self.load_state_dict(sd)
