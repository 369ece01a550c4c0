"""``causal_dot_product`` on MI355X: same surface as the reference module
``fast_transformers/causal_product/__init__.py``.

* ``CausalDotProduct`` is a ``torch.autograd.Function`` with the class-level
  dispatch tables ``dot`` / ``dot_backward`` keyed by ``device.type``
  (reference ``__init__.py:23-30``).  ROCm PyTorch reports ``"cuda"`` for an AMD
  GPU, so the HIP kernels register under that key.  The ``"cpu"`` entry is a small
  chunked implementation of its own for CPU tensors (plain torch matmuls); the GPU entry
  never falls back to it: without the HIP library a GPU tensor raises.
* The native functions keep the reference's in-place calling convention
  (``causal_product_cpu.cpp:82-87,133-141``): ``causal_dot_product(Q, K, V,
  product)`` and ``causal_dot_backward(Q, K, V, grad_out, grad_Q, grad_K,
  grad_V)`` write caller-allocated tensors and return ``None``.
* Q, K, V are float32 (as in the reference) or bfloat16 (fp32 accumulation).  The
  product is float32 in both cases (``__init__.py:41`` allocates with the default
  dtype) and the gradients have the dtype of their inputs (``__init__.py:59-61``).
"""
import torch

from .. import _native


# One scratch buffer per (device, stream), grown on demand.  The library wants the control
# block at its start zeroed before the first use and restores it after every call, so the
# buffer is allocated zero-filled once and then handed to every later call on that stream.
#
# The error word of a workspace (byte 8 of the control block) is non-zero after a call that
# was cut short.  Reading it means waiting for the GPU, so the wrapper does that only where it
# is asked for (``check_workspaces()``; after every call when FTC_CHECK=1 is set in the
# environment) or cheap (before a cached workspace is replaced by a larger one).  Between
# those it watches without waiting: at most every ten milliseconds a call leaves
# an asynchronous copy of the error word to pinned host memory behind it on its stream, and the
# next call after the copy has arrived finds the word there and raises.
_workspaces = {}
_probes = {}              # workspace key -> [pinned word, event or None]


_host_module = None


def _host():
    """The compiled binding, with this module's workspaces behind it."""
    global _host_module
    if _host_module is None:
        host = _native.host()
        host.setup(_workspaces, _probes, _make_workspace, _watch, _probe, _check_if_possible)
        _host_module = host
    return _host_module


def reload_tuning():
    """Make the library read its FTC_* environment variables again (they are read once, at first
    use) and forget the workspace sizes asked for under the old values.  A debugging aid: call
    it with no work in flight."""
    _native.check(_native.load().ftc_tuning_reload(), "ftc_tuning_reload")
    _host().forget_sizes()


def _workspace(nbytes, device, stream=None):
    """The workspace of a device and stream (the current one), at least ``nbytes`` large."""
    if nbytes <= 0:
        return None, 0
    if stream is None:
        stream = torch.cuda.current_stream(device).cuda_stream
    key = (device.index if device.index is not None else torch.cuda.current_device(), stream)
    ws = _workspaces.get(key)
    if ws is None or ws.numel() < nbytes:
        ws = _make_workspace(nbytes, key)
    return ws, ws.numel()


def _make_workspace(nbytes, key):
    if key in _workspaces:
        check_workspaces()  # the old buffer's last word on the calls made with it
    ws = torch.zeros(max(nbytes, 1 << 20), dtype=torch.uint8, device=torch.device("cuda", key[0]))
    _workspaces[key] = ws
    _probes.pop(key, None)
    return ws


def _watch(key, ws):
    """Look at a finished probe of this workspace, if there is one; otherwise nothing."""
    probe = _probes.get(key)
    if probe is None or probe[1] is None:
        return
    if not torch.cuda.is_current_stream_capturing() and probe[1].query():
        probe[1] = None
        if int(probe[0].item()) != 0:
            check_workspaces()   # synchronises, resets the control block and raises


def _probe(key, ws):
    """Leave a probe behind the call just made when the last one has been read."""
    probe = _probes.get(key)
    if (probe is not None and probe[1] is not None) or torch.cuda.is_current_stream_capturing():
        return
    if probe is None:
        probe = _probes[key] = [torch.zeros(1, dtype=torch.int32).pin_memory(), None]
    probe[0].copy_(ws[8:12].view(torch.int32), non_blocking=True)
    ev = torch.cuda.Event()
    ev.record()
    probe[1] = ev


def _check_if_possible():
    """After every call under FTC_CHECK.  The check synchronises, which a capturing stream does
    not allow: a captured call is checked by the first eager call after the replays, or by
    check_workspaces()."""
    if not torch.cuda.is_current_stream_capturing():
        check_workspaces()


def workspace_error_words():
    """Error word of every cached workspace (synchronises).  All zero unless a wavefront
    gave up waiting for another one, which a correct launch never does."""
    # (a copy: reading a word waits, and another thread may add its workspace meanwhile)
    return {key: int(ws[8:12].view(torch.int32).item()) for key, ws in _workspaces.copy().items()}


def check_workspaces():
    """Synchronise and raise if any cached workspace reports that a call was cut short.  The
    control block of such a workspace is cleared first (``ftc_workspace_reset``, on the current
    stream of its device once that device is idle: the stream the workspace was cached for may
    be gone by now), so calls made after the exception start from a clean workspace again: a
    control block left non-zero would make every later call on it stop early with its outputs
    unwritten."""
    bad = {key: word for key, word in workspace_error_words().items() if word != 0}
    if not bad:
        return
    lib = _native.load()
    for (device_index, stream) in bad:
        ws = _workspaces[(device_index, stream)]
        with torch.cuda.device(device_index):
            torch.cuda.synchronize()
            _native.check(lib.ftc_workspace_reset(ws.data_ptr(), ws.numel(),
                                                  torch.cuda.current_stream().cuda_stream),
                          "ftc_workspace_reset")
            torch.cuda.synchronize()
        _probes.pop((device_index, stream), None)
    raise RuntimeError("causal_dot_product: a call was cut short on workspace(s) %s "
                       "(error words %s); its outputs are not valid.  The workspaces have "
                       "been reset." % (sorted(bad), [bad[k] for k in sorted(bad)]))


def causal_dot_product_hip(queries, keys, values, product):
    """In-place forward; replaces the reference's native ``causal_dot_product``
    (``causal_product_cuda.cu:1273-1285``).  Enqueued on the current stream."""
    _host().forward(queries, keys, values, product)


def causal_dot_product_with_state(queries, keys, values, initial_state=None,
                                  return_state=True):
    """The product of a piece of a sequence, started from ``initial_state`` (``(N, H, E, M)``
    float32, or ``None`` for zeros) and returning ``(product, final_state)``:

        S_l = initial_state + sum_{j<=l} keys_j values_j^T ;  product_l = S_l^T queries_l

    ``final_state`` is the ``S_i`` that the reference's step-wise attention keeps
    (``recurrent/attention/self_attention/linear_attention.py:63-90``), so a prompt processed
    here can be continued there, or by another call on the next piece.  Forward only (no
    autograd); enqueued on the current stream."""
    return _host().product_with_state(queries, keys, values, initial_state, return_state)


def causal_dot_backward_hip(queries, keys, values, grad_out, grad_queries, grad_keys,
                            grad_values):
    """In-place backward; replaces the reference's native ``causal_dot_backward``
    (``causal_product_cuda.cu:1438-1467``).  A gradient passed as ``None`` is skipped.
    Enqueued on the current stream."""
    _host().backward(queries, keys, values, grad_out, grad_queries, grad_keys, grad_values)


FTC_ERR_UNSUPPORTED = -2


def fused_attention_covers(queries, values, keys=None):
    """True when ``ftc_causal_linear_attention`` has a kernel for tensors of these sizes and
    element type ((N, H, L, E) queries and keys, (N, H, L, M) values)."""
    tensors = (queries, values) if keys is None else (queries, keys, values)
    if any(t.dtype != torch.float32 or t.device != queries.device for t in tensors):
        return False
    if queries.device.type != "cuda":
        return False
    if keys is not None and keys.shape[3] != queries.shape[3]:
        return False
    return queries.shape[3] in (32, 64) and values.shape[3] in (32, 64)


def causal_linear_attention_hip(queries, keys, values, key_lengths, eps, out, denominators=None):
    """In-place fused forward of causally masked linear attention with the feature map
    ``elu(x) + 1``: replaces the body of the reference module's forward
    (``attention/causal_linear_attention.py:71-104``) in one launch.  ``queries``, ``keys``:
    raw (N, H, L, E) projections; ``values``, ``out``: (N, H, L, M); ``key_lengths``: int64
    tensor of N lengths on the same device, or None; ``denominators``: None, or a float32
    (N, H, L) tensor that receives the normaliser's denominators (the backward needs them).
    Raises ``RuntimeError`` for sizes without a fused kernel (see ``fused_attention_covers``)."""
    _host().attention(queries, keys, values, key_lengths, eps, out, denominators)


def causal_linear_attention_backward_hip(queries, keys, values, key_lengths, out, denominators,
                                         grad_out, grad_queries, grad_keys, grad_values):
    """In-place backward of ``causal_linear_attention_hip``: gradients with respect to the raw
    queries, keys and values (any of the three may be None) from ``grad_out``, the forward's
    ``out`` and its ``denominators``.  Replaces what autograd does in the reference for the body
    of ``CausalLinearAttention.forward`` (``attention/causal_linear_attention.py:71-104``)."""
    _host().attention_backward(queries, keys, values, key_lengths, out, denominators, grad_out,
                               grad_queries, grad_keys, grad_values)


def encoder_forward_hip(x, layers, final_norm, heads, key_lengths):
    """A stack of post-norm encoder layers with causal linear attention and ReLU, in eval mode
    (``transformers.py:76-89,133-145`` with ``attention/attention_layer.py:96-115``): the products
    at fp32 precision on the fp16 matrix cores (``csrc/ftc_linear.hip``), the attention in its fused
    launch.  ``layers``: per layer ((weight, bias) of the query, key, value and output projections
    and of the two feed-forward products, (weight, bias, eps) of the two norms, the attention's
    eps); ``final_norm``: (weight, bias, eps) or (); ``heads``: (H, E, M)."""
    host = _host()
    native = [host.Layer(*(host.Linear(*l) for l in linears), *(host.Norm(*n) for n in norms), eps)
              for linears, norms, eps in layers]
    return host.encoder(x.contiguous(), native, host.Norm(*final_norm) if final_norm else None, *heads,
                        key_lengths)


class CausalLinearAttentionFunction(torch.autograd.Function):
    """``out = causal linear attention(queries, keys, values)`` with the feature map
    ``elu(x) + 1``, the key-length mask and the normaliser inside, one fused launch forward
    and one launch sequence backward.  Tensors in the operator's (N, H, L, X) layout (permuted
    views of the module's (N, L, H, X) tensors are fine)."""

    @staticmethod
    def forward(ctx, queries, keys, values, key_lengths, eps):
        N, H, L, _ = queries.shape
        M = values.shape[3]
        # (N, L, H, M) storage, as the module hands its result on
        out = torch.empty((N, L, H, M), device=queries.device, dtype=torch.float32).permute(0, 2, 1, 3)
        den = torch.empty((N, H, L), device=queries.device, dtype=torch.float32)
        causal_linear_attention_hip(queries, keys, values, key_lengths, eps, out, den)
        ctx.save_for_backward(queries, keys, values, out, den)
        ctx.key_lengths = key_lengths
        return out

    @staticmethod
    def backward(ctx, grad_out):
        queries, keys, values, out, den = ctx.saved_tensors
        need = ctx.needs_input_grad
        like = lambda t: torch.empty_like(t.permute(0, 2, 1, 3)).permute(0, 2, 1, 3)
        gq = like(queries) if need[0] else None
        gk = like(keys) if need[1] else None
        gv = like(values) if need[2] else None
        causal_linear_attention_backward_hip(queries, keys, values, ctx.key_lengths, out, den,
                                             grad_out, gq, gk, gv)
        return gq, gk, gv, None, None


def _cpu_args(name, *tensors):
    for t in tensors:
        if t.dim() != 4 or t.device.type != "cpu":
            raise RuntimeError("%s: expected 4-dimensional CPU tensors" % name)


def _cpu_scan(a, b, v, out, reverse, chunk=128):
    """out[l] = sum_{j<=l} (a_l . b_j) v_j on CPU tensors (reverse: j >= l), chunked along L:
    a running (D, F) state plus the masked product inside a chunk, float32 accumulation,
    written into ``out`` in place.  This is the package's own host path for CPU tensors (the
    reference keeps a ``"cpu"`` entry next to ``"cuda"``, ``__init__.py:23-30``); it shares
    nothing with the GPU path and is not a fallback for it."""
    N, H, L, D = a.shape
    state = a.new_zeros((N, H, D, v.shape[3]), dtype=torch.float32)
    starts = list(range(0, L, chunk))
    for lo in (reversed(starts) if reverse else starts):
        hi = min(L, lo + chunk)
        ac, bc, vc = (t[:, :, lo:hi].float() for t in (a, b, v))
        p = torch.matmul(ac, bc.transpose(2, 3))
        p = torch.triu(p) if reverse else torch.tril(p)
        out[:, :, lo:hi] = (torch.matmul(p, vc) + torch.matmul(ac, state)).to(out.dtype)
        state = state + torch.matmul(bc.transpose(2, 3), vc)


def causal_dot_product_cpu(queries, keys, values, product):
    """In-place forward for CPU tensors, the reference's native signature
    (``causal_product_cpu.cpp:82-87``)."""
    _cpu_args("causal_dot_product", queries, keys, values, product)
    _cpu_scan(queries, keys, values, product, False)


def causal_dot_backward_cpu(queries, keys, values, grad_out, grad_queries, grad_keys,
                            grad_values):
    """In-place backward for CPU tensors (``causal_product_cpu.cpp:133-141``): the three
    gradients are the same scan under a change of roles."""
    _cpu_args("causal_dot_backward", queries, keys, values, grad_out)
    if grad_queries is not None:
        _cpu_scan(grad_out, values, keys, grad_queries, False)
    if grad_keys is not None:
        _cpu_scan(values, grad_out, queries, grad_keys, True)
    if grad_values is not None:
        _cpu_scan(keys, queries, grad_out, grad_values, True)


class CausalDotProduct(torch.autograd.Function):
    """Compute the weighted sum of values but attending only to previous values
    (reference ``__init__.py:20-74``)."""
    dot = {
        "cpu": causal_dot_product_cpu,
        "cuda": causal_dot_product_hip,
    }
    dot_backward = {
        "cpu": causal_dot_backward_cpu,
        "cuda": causal_dot_backward_hip,
    }

    @staticmethod
    def forward(ctx, Q, K, V):
        ctx.save_for_backward(Q, K, V)

        device = Q.device
        N, H, L, _ = Q.shape
        _, _, _, M = V.shape
        # the kernels overwrite every element, so no zero fill is needed
        product = torch.empty((N, H, L, M), device=device, dtype=torch.float32)

        CausalDotProduct.dot[device.type](
            Q,
            K,
            V,
            product
        )
        return product

    @staticmethod
    def backward(ctx, grad_out):
        Q, K, V = ctx.saved_tensors

        grad_Q = torch.empty_like(Q, memory_format=torch.contiguous_format)
        grad_K = torch.empty_like(K, memory_format=torch.contiguous_format)
        grad_V = torch.empty_like(V, memory_format=torch.contiguous_format)

        CausalDotProduct.dot_backward[Q.device.type](
            Q,
            K,
            V,
            grad_out,
            grad_Q,
            grad_K,
            grad_V
        )
        return grad_Q, grad_K, grad_V


_as_defined = (CausalDotProduct.forward, CausalDotProduct.backward, causal_dot_product_hip, causal_dot_backward_hip)


def causal_dot_product(*inputs):
    """``CausalDotProduct.apply`` (the reference's alias, ``__init__.py:77-78``).  Plain tensors on the
    GPU take the same function in the C++ engine (``host/ftc_host.cpp``), which costs the host less;
    the first call, calls that are watched or transformed, and a class or tables that have been
    changed take the class."""
    if _host_module is not None and len(inputs) == 3 and not torch.compiler.is_compiling() and _as_defined == (
            CausalDotProduct.forward, CausalDotProduct.backward, CausalDotProduct.dot.get("cuda"),
            CausalDotProduct.dot_backward.get("cuda")):
        product = _host_module.dot(*inputs)
        if product is not None:
            return product
    return CausalDotProduct.apply(*inputs)
