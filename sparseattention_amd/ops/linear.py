"""`linear(layer, x)`: an nn.Linear on this package's kernels, forward and backward."""
from __future__ import annotations

import torch
import torch.nn as nn
import torch.nn.functional as F
from torch.nn.modules import module as _module
from torch.overrides import _get_current_function_mode_stack, has_torch_function
from torch.utils._device import DeviceContext

from .. import _lib


# the forwards that calls may be made without, as they are when their classes are defined or this module is loaded
FORWARDS = {cls: cls.forward for cls in (nn.Linear, nn.LayerNorm, nn.Dropout)}


def plain_module(module, cls) -> bool:
    """Whether calling `module` runs nothing but `cls`'s own forward, so that the call may be bypassed: no
    subclass, no forward set on the instance or in place of the class's, no hooks on it or on all modules."""
    return all_plain(((module, cls),))


def all_plain(modules) -> bool:
    """plain_module(m, cls) for every (m, cls): one look at the global hooks, the modules' attributes straight
    from their dictionaries."""
    if (_module._global_forward_hooks or _module._global_forward_pre_hooks or _module._global_backward_hooks
            or _module._global_backward_pre_hooks):
        return False
    for m, cls in modules:
        d = m.__dict__
        if (type(m) is not cls or cls.forward is not FORWARDS[cls] or "forward" in d or d["_forward_hooks"]
                or d["_forward_pre_hooks"] or d["_backward_hooks"] or d["_backward_pre_hooks"]):
            return False
    return True


def watched(*tensors) -> bool:
    """Whether something handles torch's own functions on these tensors itself and would miss the calls that the native
    code makes in their place: a function mode (other than a default device, which only places new tensors) or a
    tensor subclass."""
    if not has_torch_function(tensors):
        return False
    own = (torch.Tensor, nn.Parameter, type(None))
    return (any(type(m) is not DeviceContext for m in _get_current_function_mode_stack())
            or any(type(t) not in own and type(t).__torch_function__ is not torch._C._disabled_torch_function_impl for t in tensors))


def project(x: torch.Tensor, w: torch.Tensor, contract: bool = False) -> torch.Tensor:
    """x w^T, or x w with `contract`, without autograd."""
    if watched(x, w):
        return torch.matmul(x, w) if contract else F.linear(x, w)
    return _lib.ext().project(x, w, None, contract)


def weight_and_bias(layer):
    """(layer.weight, layer.bias), from the parameters' dictionary where they are there (Module.__getattr__ costs half a
    microsecond a use): sharding and pruning keep plain tensors in their places."""
    p = layer._parameters
    try:
        return p["weight"], p["bias"]
    except KeyError:
        return layer.weight, layer.bias


def _plain(layer) -> bool:
    """An nn.Linear that may be bypassed."""
    return plain_module(layer, nn.Linear)


def linear(layer, x: torch.Tensor, wide: bool = False) -> torch.Tensor:
    """layer(x).  On the GPU with 16-bit activations (or under autocast to such a type) the product runs on this
    package's kernels where they are the faster ones (csrc/hsa_linear.hip), and in training the backward
    computes the weight's and the bias's gradient in one contraction over the tokens (csrc/hsa_weight_grad.hip),
    directly in the parameters' type; everything else is the layer itself.  wide: a vocabulary projection, whose
    input gradient is a product with a long contraction (csrc/hsa_linear_long.hip)."""
    if x.is_cuda and not torch.compiler.is_compiling() and _plain(layer):
        w, b = weight_and_bias(layer)
        if not watched(x, w, b):
            y = _lib.ext().linear(x, w, b, wide)
            if y is not None:
                return y
    return layer(x)


def _bypassed_weights(layer_q, layer_k, layer_v, x, y):
    """The weights of three bias-free nn.Linear that may be bypassed for inputs x and y, or None."""
    if torch.compiler.is_compiling() or not all_plain(((layer_q, nn.Linear), (layer_k, nn.Linear), (layer_v, nn.Linear))):
        return None
    (q, bq), (k, bk), (v, bv) = weight_and_bias(layer_q), weight_and_bias(layer_k), weight_and_bias(layer_v)
    return None if bq is not None or bk is not None or bv is not None or watched(x, y, q, k, v) else (q, k, v)


def query_key_value_rows(layer_q, layer_k, layer_v, x: torch.Tensor, y: torch.Tensor):
    """(layer_q of x; layer_k, layer_v of cat([x, y], dim=1)) in training on 16-bit types (or under
    autocast to one): the rows are converted and joined in one pass, their gradients added and cut apart
    in one (csrc/hsa_rows.hip).  None where that does not apply."""
    if x.is_cuda and torch.is_grad_enabled():
        ws = _bypassed_weights(layer_q, layer_k, layer_v, x, y)
        if ws is not None:
            return _lib.ext().query_key_value_rows(x, y, *ws)
    return None


def query_key_value(layer_q, layer_k, layer_v, x: torch.Tensor, y: torch.Tensor):
    """The same without autograd: the rows stay where they are and the five products write into the joined
    results in one launch (csrc/hsa_linear.hip).  None where that does not apply."""
    if x.is_cuda:
        ws = _bypassed_weights(layer_q, layer_k, layer_v, x, y)
        if ws is not None:
            return _lib.ext().query_key_value(x, y, *ws)
    return None
