"""The reference's large-M backward fallback, on MI355X.

/root/reference/mlp_fused.md:114-146: above an M threshold the reference
leaves its fused Triton backward (whose fp32 weight-gradient atomics contend)
for library GEMMs plus one fused elementwise kernel, ``sigmoid_h_mul``
(``dz = (1 - exp(-h)) * dh``), with the weight-gradient GEMM of each layer
issued right after that layer's data-gradient GEMM ("interleaved", so that
h_l and dz_l are still in L2):

    dh2 = grad @ W3.T  ->  dw3 = h2.T @ grad
    dz2 = sigmoid(h2) * dh2  ->  dh1 = dz2 @ W2.T
    dw2 = h1.T @ dz2 ...

Here the GEMMs are rocBLAS / hipBLASLt calls through torch (data gradients in
the 16-bit element type with fp32 accumulation, weight gradients in fp32 from
the fp32 stash: sums over many rows would overflow fp16) and the elementwise
step is this library's ``mlpmk_sigmoid_h_mul`` HIP kernel, which writes dz in
fp32 for the weight-gradient GEMM and in the 16-bit type for the next
data-gradient GEMM from one read of h and dh.

The fused backward megakernel (``ops.bwd``) replaces this at every M on
MI355X -- it needs no atomics in its workspace form and was measured 4.6-21x
faster at M = 4K..1M -- so autograd uses it unless ``autograd.BACKWARD`` is
set to ``"fallback"``; this path is kept as the reference's alternative and as
a comparator.  Same arguments and results as ``ops.bwd``.

For networks no fused forward takes (fp32 tensors wider than 128, any
tensors wider than 256 or deeper than 5 layers), :func:`fwd` is the matching
forward: one launch for 16-bit networks up to 512 wide (``mlpmk_fwd_layers``),
else fp32 library GEMMs and this library's fp32 softplus kernel
(``mlpmk_softplus_f32``); :func:`bwd` then runs the backward (every GEMM in
fp32 for fp32 tensors).
"""
from __future__ import annotations

import ctypes

import torch
import torch.nn.functional as F

from . import _lib
from .ops import _check, _elem_code, _fwd_code, _launch


def sigmoid_h_mul(h, dh, dz16_dtype=None):
    """``dz = dh * (1 - exp(-h))`` (``mlpmk_sigmoid_h_mul``): ``h`` fp32, ``dh``
    fp32 / fp16 / bf16, same shape, contiguous, on one GPU.  Returns the fp32
    ``dz`` and, when ``dz16_dtype`` is given, ``dz`` in that 16-bit type."""
    if h.dtype != torch.float32 or h.shape != dh.shape:
        raise ValueError("h must be fp32 and shaped like dh")
    if not (h.is_contiguous() and dh.is_contiguous()) or h.device != dh.device or h.device.type != "cuda":
        raise ValueError("h and dh must be contiguous tensors on one GPU")
    dh_code = _lib.DTYPE_F32 if dh.dtype == torch.float32 else _elem_code(dh.dtype, "dh")
    dz32 = torch.empty_like(h)
    dz16 = torch.empty_like(h, dtype=dz16_dtype) if dz16_dtype is not None else None
    dz16_code = _elem_code(dz16_dtype, "dz16") if dz16_dtype is not None else _lib.DTYPE_F16
    lib = _lib.get()
    rc = _launch(h.device, lib.mlpmk_sigmoid_h_mul, h.data_ptr(), dh.data_ptr(), dh_code, dz32.data_ptr(),
                 dz16.data_ptr() if dz16 is not None else None, dz16_code, h.numel())
    _check("mlpmk_sigmoid_h_mul", rc)
    return (dz32, dz16) if dz16_dtype is not None else dz32


def softplus_f32(z, out=None):
    """``h = softplus(z)`` elementwise in fp32 (``mlpmk_softplus_f32``: torch's
    softplus with beta 1 and threshold 20, kernel.py:168-171).  ``z`` fp32,
    contiguous, on a GPU; ``out`` may be ``z`` itself (default: a new tensor)."""
    if z.dtype != torch.float32 or not z.is_contiguous() or z.device.type != "cuda":
        raise ValueError("z must be a contiguous fp32 tensor on a GPU")
    h = torch.empty_like(z) if out is None else out
    if h.shape != z.shape or h.dtype != torch.float32 or not h.is_contiguous() or h.device != z.device:
        raise ValueError("out must be a contiguous fp32 tensor shaped like z on its GPU")
    rc = _launch(z.device, _lib.get().mlpmk_softplus_f32, z.data_ptr(), h.data_ptr(), z.numel())
    _check("mlpmk_softplus_f32", rc)
    return h


_layers_ws = {}  # (widths, dtype) -> workspace bytes of mlpmk_fwd_layers, -1 where it takes no such network


def _layers_workspace(dims, dtype):
    key = (dims, dtype)
    n = _layers_ws.get(key)
    if n is None:
        out = ctypes.c_int64(-1)
        if dtype != torch.float32 and min(dims) > 0:  # (a layer of no features is the library GEMMs' to run)
            rc = _lib.get().mlpmk_fwd_layers_workspace_size(len(dims) - 1, _lib.dims_array(dims), _fwd_code(dtype),
                                                            ctypes.byref(out))
            if rc not in (0, 2):  # MLPMK_ERR_UNSUPPORTED_SHAPE: -1 stays
                _check("mlpmk_fwd_layers_workspace_size", rc)
        n = _layers_ws[key] = out.value
    return n


def _gemms_faster(dims, M):
    """True where the library GEMMs run a narrow 16-bit network sooner than the
    one-launch kernel.  That kernel spends 0.12 ns per row on each layer of at
    most 64 features, whatever their number (6 of its 8 waves have no feature
    group); the GEMM route moves about 28 bytes per row and hidden feature and
    10 per input and output feature, at 2 to 4 TB/s from a few hundred
    thousand rows on (below, its launches take longer: 38 us a layer).
    Kernel / GEMMs in us, bytes per layer in brackets: 8-8-1 [157] 350,000 rows
    99 / 83, 1,200,000 318 / 210; 8-8-8-8 [203] 350,000 136 / 138, 500,000 189 /
    172, 1,200,000 443 / 350; 24-8-8-24 [309] 500,000 193 / 245, 2,097,152 772 /
    700; 63-8-8-1 [363] 2,097,152 1042 / 737; 7 x 16 [427] 500,000 383 / 426,
    2,097,152 1561 / 1535; 16-24-16 [496] 1,048,576 257 / 270, 4,194,304 1007 /
    1126."""
    if M < 400000:
        return False
    moved = 10 * (dims[0] + dims[-1]) + 28 * sum(dims[1:-1])
    return moved < (400 if M >= 1 << 20 else 300) * (len(dims) - 1)


def _fwd_layers(x, weights, stash):
    """:func:`fwd` through ``mlpmk_fwd_layers``, or None where that kernel does
    not take the call (fp32 tensors, widths above 512, more than 8 layers,
    hidden widths that are not multiples of 8, tensors off a 16-byte
    boundary) or is not the faster route (``_gemms_faster``).  An input width
    that is not a multiple of 8 is padded with zero columns of x and zero rows
    of W_1, which add nothing to the product."""
    if x.dim() != 2 or any(w.dim() != 2 for w in weights):
        return None
    dims = (int(x.shape[1]),) + tuple(int(w.shape[1]) for w in weights)
    if x.device.type != "cuda" or any(w.device != x.device for w in weights) or _gemms_faster(dims, int(x.shape[0])):
        return None
    pad = -dims[0] % 8
    dims = (dims[0] + pad,) + dims[1:]
    nbytes = _layers_workspace(dims, x.dtype)
    if nbytes < 0 or any(tuple(w.shape) != (k, n) for w, k, n in zip(weights, (dims[0] - pad,) + dims[1:], dims[1:])):
        return None
    x, weights = x.contiguous(), [w.contiguous() for w in weights]
    if pad:
        x, weights[0] = F.pad(x, (0, pad)), F.pad(weights[0], (0, 0, 0, pad))
    if x.data_ptr() % 16 or any(w.data_ptr() % 16 for w in weights):
        return None
    dev, M = x.device, int(x.shape[0])
    out = torch.empty((M, dims[-1]), dtype=x.dtype, device=dev)
    hs = [torch.empty((M, d), dtype=torch.float32, device=dev) for d in dims[1:-1]] if stash else None
    ws = torch.empty(nbytes, dtype=torch.uint8, device=dev)
    L = len(weights)
    rc = _launch(dev, _lib.get().mlpmk_fwd_layers, L, _lib.dims_array(dims), _fwd_code(x.dtype), x.data_ptr(),
                 (_lib.c_void_p * L)(*[w.data_ptr() for w in weights]), out.data_ptr(),
                 (_lib.c_void_p * (L - 1))(*[h.data_ptr() for h in hs]) if stash else None, ws.data_ptr(), nbytes, M)
    _check("mlpmk_fwd_layers", rc)
    return (out, hs) if stash else out


def fwd(x, weights, stash=False):
    """Forward for the networks no megakernel takes: fp32 tensors wider than
    128, any tensors wider than 256, more than 5 layers, hidden widths that
    are not multiples of 16.  16-bit networks up to 512 wide and 8 layers deep
    run in one launch (``mlpmk_fwd_layers``, after one that packs the weights;
    128-512-512-128 in fp16 at 16,384 rows 182 us layer by layer, 26 us), but
    for the narrowest of many rows (``_gemms_faster``).
    The others run layer by layer: ``z = a @ W_l``
    as an fp32 library GEMM (rocBLAS / hipBLASLt through torch; 16-bit
    values are exact in fp32, so this is the fused kernels' fp32
    accumulation), then the fp32 softplus kernel on every hidden layer.
    Either way the hidden h is
    rounded to the tensor format before the next layer as the
    reference's kernel rounds its h (kernel.py:110,117).  The reference's
    kernels take any width (kernel.py:60-63; INPUT_DTYPE = fp32,
    mlp_fused.md:159-166).  Returns ``out`` in x's dtype, or ``(out, [h1 ..
    h_{L-1}])`` with the fp32 stash that :func:`bwd` reads."""
    dt = x.dtype
    if dt not in (torch.float32, torch.float16, torch.bfloat16) or any(w.dtype != dt for w in weights):
        raise ValueError("x and the weights must share one of fp32, fp16 or bf16")
    res = _fwd_layers(x, weights, stash)
    if res is not None:
        return res
    a = x.contiguous() if dt == torch.float32 else x.float()
    hs = []
    with torch.autocast("cuda", enabled=False):  # the GEMMs stay fp32 under a caller's autocast
        for i, w in enumerate(weights):
            z = a @ (w.contiguous() if dt == torch.float32 else w.float())
            if i + 1 < len(weights):
                h = softplus_f32(z, out=z)
                hs.append(h)
                a = h if dt == torch.float32 else h.to(dt).float()
            else:
                a = z if dt == torch.float32 else z.to(dt)
    return (a, hs) if stash else a


def bwd(x, weights, hs, dout, dws, dx=None):
    """Gradients of ``out = MLP(x)`` from the fp32 stash ``hs`` = [h1 ..
    h_{L-1}]: ``dws[l] += h_l^T dz_l`` (``h_0 = x``) and, if ``dx`` is given,
    ``dx = dz_0 W_0^T``, in the interleaved order of mlp_fused.md:139-145.
    ``dout`` may be a broadcast row (stride 0), as ``loss = out.sum()``
    gives."""
    L = len(weights)
    if len(hs) != L - 1 or any(h is None for h in hs):
        raise ValueError("the fallback backward reads every hidden activation from the stash (no recompute)")
    with torch.autocast("cuda", enabled=False):  # GEMMs in the types below, whatever the caller's autocast
        return _bwd(x, weights, hs, dout, dws, dx)


def _bwd(x, weights, hs, dout, dws, dx):
    L = len(weights)
    dt = x.dtype
    dz16 = dout.to(dt).contiguous() if dout.stride(0) != 0 else dout[:1].to(dt).expand_as(dout).contiguous()
    dz32 = dz16.float()
    f32 = dt == torch.float32  # fp32 tensors: every GEMM in fp32
    for l in range(L - 1, -1, -1):
        need_dh = l > 0 or dx is not None
        if need_dh:
            dh = dz16 @ weights[l].t().contiguous()  # data gradient: 16-bit GEMM, fp32 accumulation
        a = hs[l - 1] if l > 0 else x.float()
        dws[l].add_(a.t() @ dz32)  # weight gradient: fp32 GEMM, right after (interleaved)
        if l > 0 and f32:
            dz32 = dz16 = sigmoid_h_mul(hs[l - 1], dh.contiguous())
        elif l > 0:
            dz32, dz16 = sigmoid_h_mul(hs[l - 1], dh.contiguous(), dz16_dtype=dt)
        elif dx is not None:
            dx.copy_(dh)
    return dws, dx
