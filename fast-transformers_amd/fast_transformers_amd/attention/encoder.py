"""Encoder blocks around ``CausalLinearAttention`` (for the 8-layer encoder workload).

Own counterparts of ``fast_transformers/attention/attention_layer.py:44-115`` (Q/K/V/out
projections around an inner attention) and ``fast_transformers/transformers.py:21-145``
(post-norm encoder layer, stack with optional final norm).  Parameter names match the
reference modules so that a reference ``state_dict`` loads unchanged.  Plain ``torch.nn``:
the custom kernels are inside the inner attention -- and, for a whole encoder of plain layers in
inference, in its matrix products and norms as well (``TransformerEncoder._fused_forward``).
"""
import torch
import torch.nn.functional as F
from torch.nn import Dropout, LayerNorm, Linear, Module, ModuleList, Parameter
from torch.utils._device import DeviceContext

from ..causal_product import encoder_forward_hip
from ..masking import FullMask, LengthMask, TriangularCausalMask
from .causal_linear_attention import CausalLinearAttention, ActivationFunctionFeatureMap, _elu_plus_one


class AttentionLayer(Module):
    """Project to multi-head queries/keys/values, run the inner attention, project back
    (``attention_layer.py:44-115``)."""

    def __init__(self, attention, d_model, n_heads, d_keys=None, d_values=None,
                 d_model_keys=None):
        super().__init__()
        d_keys = d_keys or (d_model // n_heads)
        d_values = d_values or (d_model // n_heads)
        d_model_keys = d_model_keys or d_model
        self.inner_attention = attention
        self.query_projection = Linear(d_model, d_keys * n_heads)
        self.key_projection = Linear(d_model_keys, d_keys * n_heads)
        self.value_projection = Linear(d_model_keys, d_values * n_heads)
        self.out_projection = Linear(d_values * n_heads, d_model)
        self.n_heads = n_heads

    def forward(self, queries, keys, values, attn_mask, query_lengths, key_lengths):
        N, L, _ = queries.shape
        S = keys.shape[1]
        H = self.n_heads
        q = self.query_projection(queries).view(N, L, H, -1)
        k = self.key_projection(keys).view(N, S, H, -1)
        v = self.value_projection(values).view(N, S, H, -1)
        new_values = self.inner_attention(q, k, v, attn_mask, query_lengths,
                                          key_lengths).reshape(N, L, -1)
        return self.out_projection(new_values)


class TransformerEncoderLayer(Module):
    """Self attention + feed-forward with skip connections, post-norm
    (``transformers.py:21-89``)."""

    def __init__(self, attention, d_model, d_ff=None, dropout=0.1, activation="relu"):
        super().__init__()
        d_ff = d_ff or 4 * d_model
        self.attention = attention
        self.linear1 = Linear(d_model, d_ff)
        self.linear2 = Linear(d_ff, d_model)
        self.norm1 = LayerNorm(d_model)
        self.norm2 = LayerNorm(d_model)
        self.dropout = Dropout(dropout)
        self.activation = getattr(F, activation)

    def forward(self, x, attn_mask=None, length_mask=None):
        N, L = x.shape[0], x.shape[1]
        attn_mask = attn_mask or FullMask(L, device=x.device)
        length_mask = length_mask or LengthMask(x.new_full((N,), L, dtype=torch.int64))
        x = x + self.dropout(self.attention(x, x, x, attn_mask=attn_mask,
                                            query_lengths=length_mask,
                                            key_lengths=length_mask))
        y = x = self.norm1(x)
        y = self.dropout(self.activation(self.linear1(y)))
        y = self.dropout(self.linear2(y))
        return self.norm2(x + y)


# what the native products take (ftc_linear_split, ftc_split_rows): rows, and columns or features
_MOST_ROWS, _MOST_COLUMNS = 1 << 26, 1 << 20

# what the native forward restates, as it was when this module was imported
_FORWARDS = {cls: cls.forward for cls in (Linear, LayerNorm, Dropout, AttentionLayer, TransformerEncoderLayer,
                                          CausalLinearAttention, ActivationFunctionFeatureMap)}


def _watched(module):
    # (another ``forward`` stands in for the class's: an instance's own, as offloading wrappers put it
    # there, or one that was put on the class)
    return (module._forward_hooks or module._forward_pre_hooks or "forward" in module.__dict__
            or type(module).forward is not _FORWARDS[type(module)])


def _observed():
    """True where something has to see or rewrite the single operations: a compiler or tracer, a
    functorch transform, forward-mode differentiation, a dispatch or function mode (apart from the
    default device's, which only places new tensors)."""
    return (torch.compiler.is_compiling() or torch.jit.is_tracing()
            or torch._C._functorch.peek_interpreter_stack() is not None
            or torch.autograd.forward_ad._current_level >= 0
            or torch._C._len_torch_dispatch_stack() > 0
            or any(type(mode) is not DeviceContext
                   for mode in torch.overrides._get_current_function_mode_stack()))


def _plain_tensors(x, *tensors):
    return all(t is None or (type(t) in (torch.Tensor, Parameter) and t.dtype == torch.float32 and t.device == x.device and t.is_contiguous()
                             and t.data_ptr() % 16 == 0) for t in tensors)


def _plain_linear(module, x):
    """(weight, bias) of a plain ``Linear`` whose sizes the native products take."""
    if type(module) is not Linear or _watched(module) or not _plain_tensors(x, module.weight, module.bias):
        return None
    rows, cols = module.weight.shape
    if rows % 32 or cols % 32 or cols < 64:
        return None
    return module.weight, module.bias


def _plain_norm(module, x):
    if type(module) is not LayerNorm or _watched(module) or not _plain_tensors(x, module.weight, module.bias):
        return None
    if len(module.normalized_shape) != 1 or module.normalized_shape[0] != x.shape[2] or x.shape[2] > 4096:
        return None
    return module.weight, module.bias, module.eps


def _plain_layer(layer, x):
    """(sizes of the heads, parameters) of a layer in eval mode that is made of the plain parts
    (no subclasses, hooks, other activations or feature maps), else None."""
    d = x.shape[2]
    if type(layer) is not TransformerEncoderLayer or layer.activation is not F.relu or _watched(layer):
        return None
    if layer.dropout.p > 0 and layer.dropout.training or type(layer.dropout) is not Dropout or _watched(layer.dropout):
        return None
    outer = layer.attention
    if type(outer) is not AttentionLayer or _watched(outer):
        return None
    inner = outer.inner_attention
    if type(inner) is not CausalLinearAttention or _watched(inner):
        return None
    fm = inner.feature_map
    if type(fm) is not ActivationFunctionFeatureMap or fm.activation_function is not _elu_plus_one or _watched(fm):
        return None
    linears = [_plain_linear(m, x) for m in (outer.query_projection, outer.key_projection, outer.value_projection,
                                             outer.out_projection, layer.linear1, layer.linear2)]
    norms = [_plain_norm(m, x) for m in (layer.norm1, layer.norm2)]
    if any(part is None for part in linears + norms):
        return None
    heads = outer.n_heads
    (q, k, v, o, w1, w2) = (weight for weight, _ in linears)
    if q.shape[0] % heads or v.shape[0] % heads:
        return None
    E, M = q.shape[0] // heads, v.shape[0] // heads
    if E not in (32, 64) or M not in (32, 64) or k.shape != q.shape or v.shape[0] > 4096:
        return None
    if 2 * q.shape[0] + v.shape[0] > _MOST_COLUMNS or w1.shape[0] > _MOST_COLUMNS:
        return None
    if (q.shape[1], v.shape[1], tuple(o.shape), w1.shape[1], tuple(w2.shape)) != \
            (d, d, (d, v.shape[0]), d, (d, w1.shape[0])):
        return None
    return (heads, E, M), (linears, norms, inner.eps)


class TransformerEncoder(Module):
    """A stack of encoder layers with an optional final norm (``transformers.py:92-145``)."""

    def __init__(self, layers, norm_layer=None):
        super().__init__()
        self.layers = ModuleList(layers)
        self.norm = norm_layer

    def _fused_forward(self, x, attn_mask, length_mask):
        """The whole stack in native code (``encoder_forward_hip``) where nothing has to be
        differentiated or watched and every part is the plain one; None otherwise."""
        if not (x.is_cuda and x.dtype == torch.float32 and x.dim() == 3 and x.numel() > 0) or len(self.layers) == 0:
            return None
        if x.shape[0] * x.shape[1] >= _MOST_ROWS:
            return None
        if attn_mask is None or not attn_mask.lower_triangular:
            return None
        shape = getattr(attn_mask, "shape", None)  # (a mask need not have one)
        if shape is None or shape[0] != x.shape[1]:
            return None
        if _observed() or type(x) not in (torch.Tensor, Parameter):
            return None
        if torch.is_autocast_enabled() or torch.nn.modules.module._has_any_global_hook():
            return None
        if not x.is_contiguous() or x.data_ptr() % 16:
            x = x.clone(memory_format=torch.contiguous_format)  # (the rows are read 16 bytes at a time)
        lengths = None
        if length_mask is not None:
            lengths = getattr(length_mask, "lengths", None)
            if lengths is None:
                return None
            lengths = lengths.to(device=x.device, dtype=torch.int64).contiguous()
        layers = [_plain_layer(layer, x) for layer in self.layers]
        if any(layer is None or layer[0] != layers[0][0] for layer in layers):
            return None
        norm = _plain_norm(self.norm, x) if self.norm is not None else ()
        if norm is None or (torch.is_grad_enabled() and (
                x.requires_grad or any(p.requires_grad for p in self.parameters()))):
            return None
        return encoder_forward_hip(x, [layer[1] for layer in layers], norm, layers[0][0], lengths)

    def forward(self, x, attn_mask=None, length_mask=None):
        fused = self._fused_forward(x, attn_mask, length_mask)
        if fused is not None:
            return fused
        N, L = x.shape[0], x.shape[1]
        attn_mask = attn_mask or FullMask(L, device=x.device)
        length_mask = length_mask or LengthMask(x.new_full((N,), L, dtype=torch.int64))
        for layer in self.layers:
            x = layer(x, attn_mask=attn_mask, length_mask=length_mask)
        if self.norm is not None:
            x = self.norm(x)
        return x


def build_causal_linear_encoder(n_layers=8, n_heads=8, query_dimensions=64,
                                value_dimensions=64, feed_forward_dimensions=1024,
                                dropout=0.1, activation="relu", final_normalization=True):
    """What ``TransformerEncoderBuilder.from_kwargs(attention_type="causal-linear", ...).get()``
    assembles (``builders/transformer_builders.py:219-251``): d_model = n_heads *
    value_dimensions, one ``AttentionLayer(CausalLinearAttention)`` per layer, final
    LayerNorm.  The caller passes ``attn_mask=TriangularCausalMask(L)``."""
    d_model = n_heads * value_dimensions
    layers = [
        TransformerEncoderLayer(
            AttentionLayer(CausalLinearAttention(query_dimensions), d_model, n_heads,
                           d_keys=query_dimensions, d_values=value_dimensions),
            d_model, feed_forward_dimensions, dropout, activation)
        for _ in range(n_layers)
    ]
    return TransformerEncoder(layers, LayerNorm(d_model) if final_normalization else None)


__all__ = ["AttentionLayer", "TransformerEncoderLayer", "TransformerEncoder",
           "build_causal_linear_encoder", "TriangularCausalMask", "LengthMask", "FullMask"]
