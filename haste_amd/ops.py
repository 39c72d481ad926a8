"""Op-level interface: the functions the reference exposes from its PyTorch binding
(`haste_pytorch_lib.<cell>_forward / <cell>_backward`, reference
frameworks/pytorch/{lstm,gru,indrnn,layer_norm_lstm,layer_norm_gru,layer_norm_indrnn}.cc),
with the same argument order, allocation protocol and return tuples, implemented by
calls into libhaste_hip.so.  Tensors are float32 or float64, for the GRU also float16 (all tensors of a call alike),
contiguous, on the GPU; torch is used only to allocate device memory and to name the
current stream.
"""
import torch

from . import lib


def _check(*tensors):
    # reference frameworks/pytorch/support.h:20-22 (CHECK_INPUT)
    for t in tensors:
        if t is None:
            continue
        if not t.is_cuda:
            raise ValueError("tensor must be a GPU tensor")
        if not t.is_contiguous():
            raise ValueError("tensor must be contiguous")
        if t.dtype not in _SUFFIX and t.numel():
            raise ValueError("only float32, float64 and (GRU) float16 are implemented")


_SUFFIX = {torch.float32: "_f32", torch.float64: "_f64", torch.float16: "_f16"}


def _call(entry, *args):
    """Calls `entry` + "_f32" / "_f64" according to the tensors among `args`, which must all
    have one dtype (the reference's bindings dispatch the same way, AT_DISPATCH_FLOATING_TYPES,
    frameworks/pytorch/lstm.cc:65)."""
    dtype = None
    values = []
    for a in args:  # (one pass over them: a single step's call costs as much on the host as on the GPU)
        if isinstance(a, torch.Tensor):
            if a.dtype is not dtype and a.numel():
                if dtype is not None:
                    dtypes = {t.dtype for t in args if isinstance(t, torch.Tensor) and t.numel()}
                    raise ValueError("all tensors of a call must have the same dtype, got %s" % sorted(map(str, dtypes)))
                dtype = a.dtype
            a = a.data_ptr()
        values.append(a)
    if dtype is None:
        raise ValueError("all tensors of a call must have the same dtype, got []")
    name = entry + _SUFFIX[dtype]
    fn = lib.entry(name)
    if fn is None:
        # as in the reference, half exists for the GRU only (lib/gru_forward_gpu.cu.cc:373)
        raise ValueError("%s is not implemented" % name)
    lib.invoke(name, fn, values)


def stream_status(stream=None):
    """After the caller has synchronized `stream` (default: the current stream): raises
    lib.HasteHipError when a persistent kernel launched on it gave up a bounded wait (its
    outputs, and those of library kernels queued behind it, are invalid); see
    haste_hip_stream_status in include/haste_hip.h."""
    import ctypes
    handle = lib.load()
    if stream is None:
        stream = torch.cuda.current_stream().cuda_stream
    handle.haste_hip_stream_status.restype = ctypes.c_int
    rc = handle.haste_hip_stream_status(ctypes.c_void_p(stream))
    if rc != 0:
        raise lib.HasteHipError(rc, "haste_hip_stream_status")


def workspace_bytes(time_steps, batch_size, input_size, hidden_size, half_gru=False):
    """Upper bound of the scratch memory any cell needs for these sizes on the current device
    (half_gru: the GRU on half tensors, which also stages fp32 copies of its tensors there)."""
    import ctypes
    handle = lib.load()
    fn = handle.haste_hip_gru_half_workspace_bytes if half_gru else handle.haste_hip_workspace_bytes
    fn.restype = ctypes.c_size_t
    fn.argtypes = [ctypes.c_int] * 4
    return int(fn(time_steps, batch_size, input_size, hidden_size))


def set_workspace(buffer, stream=None):
    """Lends the library `buffer` (a contiguous GPU tensor from torch's allocator, which the
    caller keeps alive and leaves alone) as the scratch memory of `stream` (default: the current
    stream); None takes it back.  With a lent buffer the ops allocate, free and synchronize
    nothing themselves, so they can be recorded into a HIP graph."""
    import ctypes
    handle = lib.load()
    if stream is None:
        stream = torch.cuda.current_stream().cuda_stream
    handle.haste_hip_set_workspace.restype = ctypes.c_int
    handle.haste_hip_set_workspace.argtypes = [ctypes.c_void_p, ctypes.c_void_p, ctypes.c_size_t]
    if buffer is None:
        rc = handle.haste_hip_set_workspace(ctypes.c_void_p(stream), None, 0)
    else:
        if not (buffer.is_cuda and buffer.is_contiguous()):
            raise ValueError("the workspace must be a contiguous GPU tensor")
        rc = handle.haste_hip_set_workspace(ctypes.c_void_p(stream), ctypes.c_void_p(buffer.data_ptr()),
                                            buffer.numel() * buffer.element_size())
    if rc != 0:
        raise lib.HasteHipError(rc, "haste_hip_set_workspace")


def workspace_high_water(stream=None):
    """Bytes of scratch memory the calls made on `stream` so far have needed (what to lend for
    a replay of the same calls)."""
    import ctypes
    handle = lib.load()
    if stream is None:
        stream = torch.cuda.current_stream().cuda_stream
    out = ctypes.c_size_t(0)
    handle.haste_hip_workspace_high_water.restype = ctypes.c_int
    rc = handle.haste_hip_workspace_high_water(ctypes.c_void_p(stream), ctypes.byref(out))
    if rc != 0:
        raise lib.HasteHipError(rc, "haste_hip_workspace_high_water")
    return int(out.value)


def _zeros(opts, *shapes):
    """Zero tensors of the given shapes carved out of one allocation: one fill kernel for all
    the accumulated outputs of a backward pass (each starts on a 256-byte boundary)."""
    sizes = [int(torch.Size(shp).numel()) for shp in shapes]
    starts, total = [], 0
    for n in sizes:
        starts.append(total)
        total += (n + 63) // 64 * 64
    flat = torch.zeros(total, **opts)
    return [flat[a:a + n].view(shp) for a, n, shp in zip(starts, sizes, shapes)]


def _given(mask):
    return mask is not None and mask.numel() > 0


def _mask_or_none(has_zoneout, zoneout_mask):
    return zoneout_mask if has_zoneout else None


def _first_states(T, N, H, first, opts):
    """State sequences [T+1,N,H], one per tensor in `first`, with slot 0 preset to it (None: zeros) by
    one kernel for all of them."""
    seqs = [torch.empty(T + 1, N, H, **opts) for _ in first]
    given = [(q[0], f) for q, f in zip(seqs, first) if f is not None]
    empty = [q[0] for q, f in zip(seqs, first) if f is None]
    if given:
        torch._foreach_copy_([q for q, _ in given], [f for _, f in given])
    if empty:
        torch._foreach_zero_(empty)
    return seqs


def _upstream(grad, T, like):
    """The address a backward entry point takes for the gradients of the states: it expects
    [T+1,N,H] and reads slots 1 .. T, so gradients [T,N,H] of the states after each step are handed
    over as they are, with the address of the slot before them.  like: one state, [N,H]."""
    if grad is None:
        return None
    if grad.dtype != like.dtype or grad.device != like.device:
        raise ValueError("all tensors of a call must have the same dtype and device, got %s on %s and %s on %s"
                         % (grad.dtype, grad.device, like.dtype, like.device))
    if grad.numel() >= (T + 1) * like.numel():
        return grad
    if grad.numel() != T * like.numel():
        raise ValueError("gradients of the states must be [%d,%d,%d] or [%d,%d,%d], got %s"
                         % (T + 1, *like.shape, T, *like.shape, list(grad.shape)))
    return grad.data_ptr() - like.numel() * like.element_size()


def _carried(opts, *pairs):
    """_zeros() of the shapes in `pairs` of (shape, initial value or None).  An initial value may have
    any strides (the gradient of a state that the caller transposed or summed comes that way); the
    entry points take row-major tensors."""
    for shape, start in pairs:
        if start is not None and (tuple(start.shape) != tuple(shape) or start.dtype != opts["dtype"]
                                  or start.device != opts["device"]):
            raise ValueError("gradient of the last state must be %s, %s on %s, got %s, %s on %s"
                             % (list(shape), opts["dtype"], opts["device"], list(start.shape), start.dtype, start.device))
    out = _zeros(opts, *[shape for shape, start in pairs if start is None])
    # detached: the kernels write into the copies, which a pass that is itself differentiated
    # (create_graph) would otherwise take for copies still
    return [out.pop(0) if start is None else start.detach().clone(memory_format=torch.contiguous_format)
            for _, start in pairs]


def gemm(a, b, out=None, trans_a=False, accumulate=False):
    """out[M,N] = op(a) @ b (+ out). a is [M,K], or [K,M] when trans_a."""
    _check(a, b)
    K, M = (a.shape if trans_a else (a.shape[1], a.shape[0]))
    N = b.shape[1]
    assert b.shape[0] == K
    if out is None:
        assert not accumulate
        out = torch.empty(M, N, device=a.device, dtype=a.dtype)
    _call("haste_hip_gemm", int(trans_a), M, N, K, a, a.stride(0), b, b.stride(0),
             out, out.stride(0), int(accumulate))
    return out


def transpose(a, out=None):
    """[rows, cols] -> [cols, rows] (a contiguous copy); leading dimensions of `a` beyond
    the last are folded into rows, so x[T,N,C] gives x_t[C,T,N]."""
    _check(a)
    cols = a.shape[-1]
    rows = a.numel() // cols
    if out is None:
        out = torch.empty((cols,) + tuple(a.shape[:-1]), device=a.device, dtype=a.dtype)
    _call("haste_hip_transpose", rows, cols, a, out)
    return out


def transpose3(a, b, c):
    """transpose() of three tensors in one launch: the x_t, W_t, R_t a backward pass asks its caller
    for (reference frameworks/pytorch/lstm.py:84-86)."""
    _check(a, b, c)
    outs = []
    args = []
    for m in (a, b, c):
        cols = m.shape[-1]
        out = torch.empty((cols,) + tuple(m.shape[:-1]), device=m.device, dtype=m.dtype)
        outs.append(out)
        args += [m.numel() // cols, cols, m, out]
    _call("haste_hip_transpose3", *args)
    return tuple(outs)


def _check_lengths(lengths, like):
    """The kernels read like.shape[1] 64-bit integers at the address of `lengths`."""
    if lengths.dtype != torch.int64 or lengths.device != like.device or not lengths.is_contiguous() \
            or tuple(lengths.shape) != (like.shape[1],):
        raise ValueError("lengths must be a contiguous int64 tensor [%d] on %s, got %s %s on %s"
                         % (like.shape[1], like.device, lengths.dtype, list(lengths.shape), lengths.device))


def gather_states(seqs, lengths):
    """The states [N,H] of one or two sequences [T+1,N,H] at the steps lengths[N] (int64)."""
    _check(*seqs)
    _check_lengths(lengths, seqs[0])
    if any(s.shape != seqs[0].shape or s.device != seqs[0].device for s in seqs[1:]) or len(seqs) > 2:
        raise ValueError("one or two state sequences of one shape are gathered")
    T1, N, H = seqs[0].shape
    outs = [torch.empty(N, H, device=s.device, dtype=s.dtype) for s in seqs]
    second = seqs[1:] or (None,)
    _call("haste_hip_gather_states", T1 - 1, N, H, seqs[0], second[0], lengths.data_ptr(), outs[0],
          outs[1] if len(outs) > 1 else None)
    return tuple(outs)


def state_gradients(like, grad, last, lengths):
    """Gradients [T,N,H] of the steps of a sequence `like` [T+1,N,H]: grad [T,N,H] (None: zeros) plus
    last [N,H] at the steps lengths[N] (int64; step 0, the initial state, gets none)."""
    T1, N, H = like.shape
    _check_lengths(lengths, like)
    if tuple(last.shape) != (N, H) or (grad is not None and tuple(grad.shape) != (T1 - 1, N, H)):
        raise ValueError("gradients of %s states must be [%d,%d,%d] and [%d,%d]" % (list(like.shape), T1 - 1, N, H, N, H))
    if grad is not None and grad.stride(2) != 1:
        grad = grad.contiguous()
    last = last.contiguous()
    _check(last)
    if grad is not None and grad.device != like.device:
        raise ValueError("gradients must be on %s" % like.device)
    out = torch.empty(T1 - 1, N, H, device=like.device, dtype=like.dtype)
    step, row = (0, 0) if grad is None else grad.stride()[:2]
    _call("haste_hip_state_gradients", T1 - 1, N, H, grad, step, row, last, lengths.data_ptr(), out)
    return out


# ---- LSTM (reference frameworks/pytorch/lstm.cc:31-157) ---------------------
def lstm_forward(training, zoneout_prob, x, h0, c0, kernel, recurrent_kernel, bias, zoneout_mask,
                 dropconnect_mask=None, dropconnect_scale=1.0):
    T, N, C = x.shape
    H = recurrent_kernel.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, c0, kernel, recurrent_kernel, bias, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    output, output_state = _first_states(T, N, H, (h0, c0), opts)
    cache = torch.empty(T, N, 4 * H, **opts)
    zp = float(zoneout_prob) if has_zoneout else 0.0
    mask = _mask_or_none(has_zoneout, zoneout_mask)
    if dropconnect_mask is None:
        _call("haste_hip_lstm_forward", bool(training), T, N, C, H, kernel, recurrent_kernel,
                 bias, x, output, output_state, cache, None, zp, mask)
    else:
        _check(dropconnect_mask)
        _call("haste_hip_lstm_forward_dropconnect", bool(training), T, N, C, H, kernel,
                 recurrent_kernel, bias, x, output, output_state, cache, zp, mask,
                 dropconnect_mask, float(dropconnect_scale))
    return output, output_state, cache


def lstm_backward(x_t, kernel_t, recurrent_kernel_t, bias, zoneout_mask, h, c, cache, dh_new, dc_new,
                  dh_last=None, dc_last=None):
    """dh_new, dc_new: gradients of the states, [T+1,N,H] (slot 0 is not read) or [T,N,H]; dc_new may
    be None (zeros).  dh_last, dc_last: more gradient of the last states, [N,H]."""
    C, T, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_kernel_t, bias, zoneout_mask, h, c, cache, dh_new, dc_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, dR, db, dh, dc = _carried(opts, ((C, 4 * H), None), ((H, 4 * H), None), ((4 * H,), None),
                                  ((N, H), dh_last), ((N, H), dc_last))
    _call("haste_hip_lstm_backward", T, N, C, H, kernel_t, recurrent_kernel_t, bias, x_t,
             h, c, _upstream(dh_new, T, dh), _upstream(dc_new, T, dh), dx, dW, dR, db, dh, dc, cache,
             _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dc, dW, dR, db


# ---- single LSTM steps (reference lib/haste/lstm.h:73-86,201-219; no binding of the
# reference exposes them, examples/lstm.cc:252,309 calls them from C++) ------------------
def lstm_forward_iterate(training, zoneout_prob, x, h, c, kernel, recurrent_kernel, bias,
                         zoneout_mask=None, h_out=None, c_out=None):
    """One step: x[N,C], h,c[N,H] -> h_out,c_out[N,H], v[N,4H] (activations when training)."""
    N, C = x.shape
    H = recurrent_kernel.shape[0]
    _check(x, h, c, kernel, recurrent_kernel, bias)
    h_out = torch.empty_like(h) if h_out is None else h_out
    c_out = torch.empty_like(c) if c_out is None else c_out
    v = torch.empty(N, 4 * H, device=x.device, dtype=x.dtype)
    has_zoneout = bool(zoneout_prob) and zoneout_mask is not None and zoneout_mask.numel() > 0
    _call("haste_hip_lstm_forward_iterate", bool(training), N, C, H, kernel, recurrent_kernel,
             bias, x, h, c, h_out, c_out, v, None, float(zoneout_prob) if has_zoneout else 0.0,
             zoneout_mask if has_zoneout else None)
    return h_out, c_out, v


def lstm_backward_iterate(x_t, kernel_t, recurrent_kernel_t, bias, h, c, c_new, dh_new, dc_new, v,
                          dW, dR, db, dh, dc, zoneout_mask=None):
    """One reverse step: x_t[C,N]; h,c = states before the step, c_new = cell state after it;
    dW, dR, db are accumulated into, dh, dc updated in place, v consumed.  Returns dx[N,C]."""
    C, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    _check(x_t, kernel_t, recurrent_kernel_t, bias, h, c, c_new, dh_new, dc_new, v, dW, dR, db, dh, dc)
    dx = torch.empty(N, C, device=x_t.device, dtype=x_t.dtype)
    has_zoneout = zoneout_mask is not None and zoneout_mask.numel() > 0
    _call("haste_hip_lstm_backward_iterate", N, C, H, kernel_t, recurrent_kernel_t, bias, x_t,
             h, c, c_new, dh_new, dc_new, dx, dW, dR, db, dh, dc, v,
             zoneout_mask if has_zoneout else None)
    return dx


# ---- single GRU steps (reference lib/haste/gru.h:72-84,172-189) -------------------------
def gru_forward_iterate(training, zoneout_prob, x, h, kernel, recurrent_kernel, bias,
                        recurrent_bias, zoneout_mask=None, h_out=None):
    N, C = x.shape
    H = recurrent_kernel.shape[0]
    _check(x, h, kernel, recurrent_kernel, bias, recurrent_bias)
    h_out = torch.empty_like(h) if h_out is None else h_out
    v = torch.empty(N, 4 * H, device=x.device, dtype=x.dtype)
    tmp_Wx = torch.empty(N, 3 * H, device=x.device, dtype=x.dtype)
    has_zoneout = bool(zoneout_prob) and zoneout_mask is not None and zoneout_mask.numel() > 0
    _call("haste_hip_gru_forward_iterate", bool(training), N, C, H, kernel, recurrent_kernel,
             bias, recurrent_bias, x, h, h_out, v, tmp_Wx, None,
             float(zoneout_prob) if has_zoneout else 0.0, zoneout_mask if has_zoneout else None)
    return h_out, v


def gru_backward_iterate(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, h, v, dh_new,
                         dW, dR, dbx, dbr, dh, zoneout_mask=None):
    C, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    _check(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, h, v, dh_new, dW, dR, dbx, dbr, dh)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(N, C, **opts)
    dp = torch.empty(N, 3 * H, **opts)
    dq = torch.empty(N, 3 * H, **opts)
    has_zoneout = zoneout_mask is not None and zoneout_mask.numel() > 0
    _call("haste_hip_gru_backward_iterate", N, C, H, kernel_t, recurrent_kernel_t, bias,
             recurrent_bias, x_t, h, v, dh_new, dx, dW, dR, dbx, dbr, dh, dp, dq,
             zoneout_mask if has_zoneout else None)
    return dx


# ---- GRU (reference frameworks/pytorch/gru.cc:30-163) -----------------------
def gru_forward(training, zoneout_prob, x, h0, kernel, recurrent_kernel, bias, recurrent_bias,
                zoneout_mask, dropconnect_mask=None, dropconnect_scale=1.0):
    T, N, C = x.shape
    H = recurrent_kernel.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, kernel, recurrent_kernel, bias, recurrent_bias, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    (output,) = _first_states(T, N, H, (h0,), opts)
    cache = torch.empty(T, N, 4 * H, **opts)
    tmp_Wx = torch.empty(T, N, 3 * H, **opts)
    zp = float(zoneout_prob) if has_zoneout else 0.0
    mask = _mask_or_none(has_zoneout, zoneout_mask)
    if dropconnect_mask is None:
        _call("haste_hip_gru_forward", bool(training), T, N, C, H, kernel, recurrent_kernel,
                 bias, recurrent_bias, x, output, cache if training else None, tmp_Wx, None, zp, mask)
    else:
        _check(dropconnect_mask)
        _call("haste_hip_gru_forward_dropconnect", bool(training), T, N, C, H, kernel,
                 recurrent_kernel, bias, recurrent_bias, x, output, cache if training else None,
                 tmp_Wx, zp, mask, dropconnect_mask, float(dropconnect_scale))
    return output, cache


def gru_backward(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, zoneout_mask, h, cache,
                 dh_new, dh_last=None):
    C, T, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, zoneout_mask, h, cache, dh_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, dR, dbx, dbr, dh = _carried(opts, ((C, 3 * H), None), ((H, 3 * H), None), ((3 * H,), None),
                                    ((3 * H,), None), ((N, H), dh_last))
    dp = torch.empty(T, N, 3 * H, **opts)
    dq = torch.empty(T, N, 3 * H, **opts)
    _call("haste_hip_gru_backward", T, N, C, H, kernel_t, recurrent_kernel_t, bias,
             recurrent_bias, x_t, h, cache, _upstream(dh_new, T, dh), dx, dW, dR, dbx, dbr, dh, dp, dq,
             _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dW, dR, dbx, dbr


# ---- Layer norm (reference lib/haste/layer_norm.h) ---------------------------
def layer_norm_forward(x, gamma, beta=None):
    _check(x, gamma)
    rows, dim = x.numel() // x.shape[-1], x.shape[-1]
    y = torch.empty_like(x)
    cache = torch.empty(rows, 2, device=x.device, dtype=x.dtype)
    _call("haste_hip_layer_norm_forward", rows, dim, gamma, beta, x, y, cache)
    return y, cache


def layer_norm_backward(x, gamma, dy, cache=None, with_beta=True, in_place=False):
    _check(x, gamma, dy)
    rows, dim = x.numel() // x.shape[-1], x.shape[-1]
    dx = dy if in_place else torch.empty_like(x)
    dgamma = torch.zeros_like(gamma)
    dbeta = torch.zeros_like(gamma) if with_beta else None
    _call("haste_hip_layer_norm_backward", rows, dim, gamma, x, dy, dx, dgamma, dbeta, cache)
    return dx, dgamma, dbeta


# ---- IndRNN (reference frameworks/pytorch/indrnn.cc:30-140) -------------------
def indrnn_forward(training, zoneout_prob, x, h0, kernel, recurrent_scale, bias, zoneout_mask):
    T, N, C = x.shape
    H = recurrent_scale.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, kernel, recurrent_scale, bias, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    (output,) = _first_states(T, N, H, (h0,), opts)
    workspace = torch.empty(T, N, H, **opts)
    _call("haste_hip_indrnn_forward", bool(training), T, N, C, H, kernel, recurrent_scale,
             bias, x, output, workspace, float(zoneout_prob) if has_zoneout else 0.0,
             _mask_or_none(has_zoneout, zoneout_mask))
    return output


def indrnn_backward(x_t, kernel_t, recurrent_scale, bias, zoneout_mask, h, dh_new, dh_last=None):
    C, T, N = x_t.shape
    H = recurrent_scale.shape[0]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_scale, bias, zoneout_mask, h, dh_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, du, db, dh = _carried(opts, ((C, H), None), ((H,), None), ((H,), None), ((N, H), dh_last))
    workspace = torch.empty(T, N, H, **opts)
    _call("haste_hip_indrnn_backward", T, N, C, H, kernel_t, recurrent_scale, bias, x_t, h,
             _upstream(dh_new, T, dh), dx, dW, du, db, dh, workspace, _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dW, du, db


# ---- LayerNorm IndRNN (reference frameworks/pytorch/layer_norm_indrnn.cc:31-174) ----
def layer_norm_indrnn_forward(training, zoneout_prob, x, h0, kernel, recurrent_scale, bias, gamma,
                              zoneout_mask):
    T, N, C = x.shape
    H = recurrent_scale.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, kernel, recurrent_scale, bias, gamma, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    (output,) = _first_states(T, N, H, (h0,), opts)
    workspace = torch.empty(T, N, H, **opts)
    act_Wx = torch.empty(T, N, H, **opts)
    act_Wx_norm_cache = torch.empty(T, N, 2, **opts)
    _call("haste_hip_layer_norm_indrnn_forward", bool(training), T, N, C, H, kernel,
             recurrent_scale, bias, x, output, workspace, act_Wx, gamma[0], act_Wx_norm_cache,
             float(zoneout_prob) if has_zoneout else 0.0, _mask_or_none(has_zoneout, zoneout_mask))
    return output, act_Wx, act_Wx_norm_cache


def layer_norm_indrnn_backward(x_t, kernel_t, recurrent_scale, bias, gamma, zoneout_mask, h, act_Wx,
                               act_Wx_norm_cache, dh_new, dh_last=None):
    C, T, N = x_t.shape
    H = recurrent_scale.shape[0]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_scale, bias, gamma, zoneout_mask, h, act_Wx, dh_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, du, db, dh = _carried(opts, ((C, H), None), ((H,), None), ((H,), None), ((N, H), dh_last))
    workspace = torch.empty(T, N, H, **opts)
    dgamma = torch.zeros_like(gamma)
    _call("haste_hip_layer_norm_indrnn_backward", T, N, C, H, kernel_t, recurrent_scale, bias,
             x_t, h, _upstream(dh_new, T, dh), dx, dW, du, db, dh, workspace, act_Wx, gamma[0], dgamma[0],
             _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dW, du, db, dgamma


# ---- LayerNorm LSTM (reference frameworks/pytorch/layer_norm_lstm.cc:31-297) ---------
def layer_norm_lstm_forward(training, zoneout_prob, x, h0, c0, kernel, recurrent_kernel, bias,
                            gamma, gamma_h, beta_h, zoneout_mask):
    T, N, C = x.shape
    H = recurrent_kernel.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, c0, kernel, recurrent_kernel, bias, gamma, gamma_h, beta_h, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    output, output_state = _first_states(T, N, H, (h0, c0), opts)
    act_Wx = torch.empty(T, N, 4 * H, **opts)
    act_Wx_norm = torch.empty(T, N, 4 * H, **opts)
    act_Wx_norm_cache = torch.empty(T, N, 2, **opts)
    act_Rh = torch.empty(T, N, 4 * H, **opts)
    act_Rh_norm_cache = torch.empty(T, N, 2, **opts)
    act_c_norm = torch.empty(T, N, H, **opts)
    act_c_norm_cache = torch.empty(T, N, 2, **opts)
    _call("haste_hip_layer_norm_lstm_forward", bool(training), T, N, C, H, kernel,
             recurrent_kernel, bias, x, output, output_state, act_Wx, None,
             gamma[0], act_Wx_norm_cache, act_Wx_norm, act_Rh, gamma[1], act_Rh_norm_cache,
             gamma_h, beta_h, act_c_norm_cache, act_c_norm,
             float(zoneout_prob) if has_zoneout else 0.0, _mask_or_none(has_zoneout, zoneout_mask))
    return (output, output_state, act_Wx, act_Wx_norm, act_Wx_norm_cache, act_Rh, act_Rh_norm_cache,
            act_c_norm, act_c_norm_cache)


def layer_norm_lstm_backward(x_t, kernel_t, recurrent_kernel_t, bias, gamma, gamma_h, beta_h,
                             zoneout_mask, h, c, act_Wx, act_Wx_norm, act_Wx_norm_cache, act_Rh,
                             act_Rh_norm_cache, act_c_norm, act_c_norm_cache, dh_new, dc_new,
                             dh_last=None, dc_last=None):
    C, T, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_kernel_t, bias, gamma, gamma_h, beta_h, zoneout_mask, h, c,
           act_Wx, act_Wx_norm, act_Wx_norm_cache, act_Rh, act_Rh_norm_cache, act_c_norm,
           act_c_norm_cache, dh_new, dc_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, dR, db, dgamma, dgamma_h, dbeta_h, dh, dc = _carried(
        opts, ((C, 4 * H), None), ((H, 4 * H), None), ((4 * H,), None), (tuple(gamma.shape), None),
        ((H,), None), ((H,), None), ((N, H), dh_last), ((N, H), dc_last))
    _call("haste_hip_layer_norm_lstm_backward", T, N, C, H, kernel_t, recurrent_kernel_t,
             bias, x_t, h, c, _upstream(dh_new, T, dh), _upstream(dc_new, T, dh), dx, dW, dR, db, dh, dc,
             act_Wx, gamma[0], dgamma[0], act_Wx_norm, act_Rh, gamma[1], dgamma[1],
             act_Rh_norm_cache, gamma_h, beta_h, dgamma_h, dbeta_h, act_c_norm_cache, act_c_norm,
             _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dc, dW, dR, db, dgamma, dgamma_h, dbeta_h


# ---- LayerNorm GRU (reference frameworks/pytorch/layer_norm_gru.cc:30-230) -----------
def layer_norm_gru_forward(training, zoneout_prob, x, h0, kernel, recurrent_kernel, bias,
                           recurrent_bias, gamma, zoneout_mask):
    T, N, C = x.shape
    H = recurrent_kernel.shape[0]
    has_zoneout = bool(zoneout_prob) and _given(zoneout_mask)
    _check(x, h0, kernel, recurrent_kernel, bias, recurrent_bias, gamma, zoneout_mask)
    opts = dict(device=x.device, dtype=x.dtype)
    (output,) = _first_states(T, N, H, (h0,), opts)
    cache = torch.empty(T, N, 4 * H, **opts)
    act_Wx = torch.empty(T, N, 3 * H, **opts)
    tmp_Wx_norm = torch.empty(T, N, 3 * H, **opts)
    act_Wx_norm_cache = torch.empty(T, N, 2, **opts)
    act_Rh = torch.empty(T, N, 3 * H, **opts)
    act_Rh_norm_cache = torch.empty(T, N, 2, **opts)
    _call("haste_hip_layer_norm_gru_forward", bool(training), T, N, C, H, kernel,
             recurrent_kernel, bias, recurrent_bias, x, output, cache if training else None,
             act_Wx, gamma[0], act_Wx_norm_cache, tmp_Wx_norm, act_Rh, gamma[1], act_Rh_norm_cache,
             None, float(zoneout_prob) if has_zoneout else 0.0,
             _mask_or_none(has_zoneout, zoneout_mask))
    return output, cache, act_Wx, act_Wx_norm_cache, act_Rh, act_Rh_norm_cache


def layer_norm_gru_backward(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, gamma,
                            zoneout_mask, h, cache, act_Wx, act_Wx_norm_cache, act_Rh,
                            act_Rh_norm_cache, dh_new, dh_last=None):
    C, T, N = x_t.shape
    H = recurrent_kernel_t.shape[1]
    has_zoneout = _given(zoneout_mask)
    _check(x_t, kernel_t, recurrent_kernel_t, bias, recurrent_bias, gamma, zoneout_mask, h, cache,
           act_Wx, act_Wx_norm_cache, act_Rh, act_Rh_norm_cache, dh_new)
    opts = dict(device=x_t.device, dtype=x_t.dtype)
    dx = torch.empty(T, N, C, **opts)
    dW, dR, dbx, dbr, dh, dgamma = _carried(opts, ((C, 3 * H), None), ((H, 3 * H), None), ((3 * H,), None),
                                            ((3 * H,), None), ((N, H), dh_last), (tuple(gamma.shape), None))
    dp = torch.empty(T, N, 3 * H, **opts)
    dq = torch.empty(T, N, 3 * H, **opts)
    _call("haste_hip_layer_norm_gru_backward", T, N, C, H, kernel_t, recurrent_kernel_t, bias,
             recurrent_bias, x_t, h, cache, _upstream(dh_new, T, dh), dx, dW, dR, dbx, dbr, dh, dp, dq,
             act_Wx, gamma[0], dgamma[0], act_Rh, gamma[1], dgamma[1], act_Rh_norm_cache,
             _mask_or_none(has_zoneout, zoneout_mask))
    return dx, dh, dW, dR, dbx, dbr, dgamma
