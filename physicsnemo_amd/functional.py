"""Tensor-level wrappers over the C ABI: one function per entry point of include/physattn.h.

Every function takes CUDA (ROCm) tensors, allocates outputs/workspace with torch and enqueues the HIP
kernels on torch's current stream.  `params` is the dict produced by
`physicsnemo_amd.physics_attention.PhysicsAttentionBase.kernel_params`.
"""
from __future__ import annotations

from ctypes import byref
from functools import lru_cache
from typing import NamedTuple

import torch

from . import _lib


class LayerDims(NamedTuple):
    B: int
    N: int
    C: int
    H: int
    D: int
    S: int
    grid_h: int = 0
    grid_w: int = 0
    conv_k: int = 0
    grid_d: int = 0
    conv_tap_major: int = 0  # 1: convolution weights are laid out (c_out, k, k[, k], c_in) instead of torch's order

    def c(self) -> _lib.PaShape:
        return _lib.PaShape.from_buffer_copy(_c_shape(self))


@lru_cache(maxsize=256)
def _c_shape(dims: LayerDims) -> bytes:  # callers get a struct of their own
    return bytes(_lib.PaShape(*dims))


_PARAM_FIELDS = [f for f, _ in _lib.PaParams._fields_]


def _c_params(params: dict) -> _lib.PaParams:
    return _lib.PaParams(*[_lib.ptr(params.get(k)) for k in _PARAM_FIELDS])


def _need_cuda(*tensors):
    for t in tensors:
        if t is not None and not t.is_cuda:
            raise RuntimeError("physicsnemo_amd runs on GPU tensors only (there is no CPU path)")
        if t is not None and not t.is_contiguous():
            raise RuntimeError("physicsnemo_amd kernels need contiguous tensors")


def query_path(dtype: torch.dtype, dims: LayerDims) -> int:
    """0 = general kernels, 1 = fused bf16 MFMA kernels, 2 = staged bf16 MFMA kernels (512-wide layers)."""
    rc = _lib.load().pa_query_path(_lib.dtype_code(dtype), byref(dims.c()))
    if rc < 0:
        _lib.check(rc, "pa_query_path")
    return rc


def project_inputs(x, params, dims: LayerDims):
    """(x_mid, fx_mid); Transolver++ parameter sets (no in_project_fx) share one projection: fx_mid is x_mid."""
    _need_cuda(x)
    lib = _lib.load()
    x_mid = torch.empty(dims.B, dims.N, dims.H * dims.D, dtype=x.dtype, device=x.device)
    fx_mid = torch.empty_like(x_mid) if params.get("in_project_fx_weight") is not None else None
    _lib.check(lib.pa_project_inputs(_lib.dtype_code(x.dtype), byref(dims.c()), byref(_c_params(params)),
                                     x.data_ptr(), x_mid.data_ptr(), _lib.ptr(fx_mid),
                                     _lib.current_stream_ptr(x.device)), "pa_project_inputs")
    return x_mid, (x_mid if fx_mid is None else fx_mid)


def slice_softmax_plus(x_mid, uniform, params, dims: LayerDims):
    """Transolver++ slice weights: learned per-point temperature and Gumbel noise from the uniform samples given."""
    _need_cuda(x_mid, uniform)
    if uniform.dtype != x_mid.dtype or uniform.shape != (dims.B, dims.N, dims.H, dims.S):
        raise ValueError("uniform samples must have the activation dtype and shape (B, N, H, S)")
    w = torch.empty(dims.B, dims.N, dims.H, dims.S, dtype=x_mid.dtype, device=x_mid.device)
    scratch = torch.empty_like(w)  # hidden layer of proj_temperature: lets both Linears run on the row GEMM kernels
    plus = _lib.PaPlusParams(*[_lib.ptr(params[k]) for k, _ in _lib.PaPlusParams._fields_])
    _lib.check(_lib.load().pa_slice_softmax_plus(_lib.dtype_code(x_mid.dtype), byref(dims.c()),
                                                 byref(_c_params(params)), byref(plus), x_mid.data_ptr(),
                                                 uniform.data_ptr(), w.data_ptr(), scratch.data_ptr(),
                                                 _lib.current_stream_ptr(x_mid.device)), "pa_slice_softmax_plus")
    return w


def slice_softmax(x_mid, params, dims: LayerDims):
    _need_cuda(x_mid)
    lib = _lib.load()
    w = torch.empty(dims.B, dims.N, dims.H, dims.S, dtype=x_mid.dtype, device=x_mid.device)
    _lib.check(lib.pa_slice_softmax(_lib.dtype_code(x_mid.dtype), byref(dims.c()), byref(_c_params(params)),
                                    x_mid.data_ptr(), w.data_ptr(), _lib.current_stream_ptr(x_mid.device)),
               "pa_slice_softmax")
    return w


def slice_reduce(w, fx_mid, dims: LayerDims):
    _need_cuda(w, fx_mid)
    lib = _lib.load()
    shape = dims.c()
    g = lib.pa_reduce_partial_count(byref(shape))
    if g < 0:
        _lib.check(int(g), "pa_reduce_partial_count")
    partials = torch.empty(g * dims.B * dims.H * dims.S * (dims.D + 1), dtype=torch.float32, device=w.device)
    tok = torch.empty(dims.B, dims.H, dims.S, dims.D, dtype=torch.float32, device=w.device)
    norm = torch.empty(dims.B, dims.H, dims.S, dtype=torch.float32, device=w.device)
    _lib.check(lib.pa_slice_reduce(_lib.dtype_code(w.dtype), byref(shape), w.data_ptr(), fx_mid.data_ptr(),
                                   partials.data_ptr(), tok.data_ptr(), norm.data_ptr(),
                                   _lib.current_stream_ptr(w.device)), "pa_slice_reduce")
    return tok, norm


def thin_tokens(x, params, dims: LayerDims):
    """(slice_token, slice_norm) of a layer whose input has few channels, in one pass over x; None where that pass does
    not serve the shape (the stages one by one do)."""
    _need_cuda(x)
    lib = _lib.load()
    shape = dims.c()
    g = lib.pa_thin_tokens_partial_count(_lib.dtype_code(x.dtype), byref(shape))
    if g < 0:
        _lib.check(int(g), "pa_thin_tokens_partial_count")
    if g == 0:
        return None
    partials = torch.empty(g * dims.B * dims.H * dims.S * (dims.D + 1), dtype=torch.float32, device=x.device)
    tok = torch.empty(dims.B, dims.H, dims.S, dims.D, dtype=torch.float32, device=x.device)
    norm = torch.empty(dims.B, dims.H, dims.S, dtype=torch.float32, device=x.device)
    _lib.check(lib.pa_thin_tokens(_lib.dtype_code(x.dtype), byref(shape), byref(_c_params(params)), x.data_ptr(),
                                  partials.data_ptr(), tok.data_ptr(), norm.data_ptr(),
                                  _lib.current_stream_ptr(x.device)), "pa_thin_tokens")
    return tok, norm


def slice_reduce_static(w, fx_mid, dims: LayerDims, out=None):
    """`slice_reduce` through the entry point that allocates nothing: the partial sums live in the library's static
    device scratch.  `out` = (slice_token, slice_norm) float32 tensors to fill (allocated here when omitted: the
    library call itself never allocates).  Calls that overlap on one GPU race on the shared scratch."""
    _need_cuda(w, fx_mid)
    tok, norm = out if out is not None else (
        torch.empty(dims.B, dims.H, dims.S, dims.D, dtype=torch.float32, device=w.device),
        torch.empty(dims.B, dims.H, dims.S, dtype=torch.float32, device=w.device))
    _lib.check(_lib.load().pa_slice_reduce_static(_lib.dtype_code(w.dtype), byref(dims.c()), w.data_ptr(),
                                                  fx_mid.data_ptr(), tok.data_ptr(), norm.data_ptr(),
                                                  _lib.current_stream_ptr(w.device)), "pa_slice_reduce_static")
    return tok, norm


def slice_attention(tok, params, dims: LayerDims):
    _need_cuda(tok)
    lib = _lib.load()
    out = torch.empty_like(tok)
    _lib.check(lib.pa_slice_attention(byref(dims.c()), byref(_c_params(params)), tok.data_ptr(), out.data_ptr(),
                                      _lib.current_stream_ptr(tok.device)), "pa_slice_attention")
    return out


def _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out):
    return _lib.PaBlockTail(_lib.ptr(residual), _lib.ptr(ln_weight), _lib.ptr(ln_bias), float(ln_eps), _lib.ptr(ln_out))


def deslice_project(w, tok_out, params, dims: LayerDims, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5,
                    return_out_x=False):
    """Returns y, or (fx_new, ln_out) when a residual / LayerNorm tail is requested; with `return_out_x` the
    desliced (B, N, H*D) input of out_linear is appended."""
    _need_cuda(w, tok_out, residual)
    lib = _lib.load()
    y = torch.empty(dims.B, dims.N, dims.C, dtype=w.dtype, device=w.device)
    scratch = torch.empty(dims.B, dims.N, dims.H * dims.D, dtype=w.dtype, device=w.device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    _lib.check(lib.pa_deslice_project(_lib.dtype_code(w.dtype), byref(dims.c()), byref(_c_params(params)),
                                      w.data_ptr(), tok_out.data_ptr(), scratch.data_ptr(), y.data_ptr(),
                                      byref(tail), _lib.current_stream_ptr(w.device)), "pa_deslice_project")
    out = y if (residual is None and ln_out is None) else (y, ln_out)
    return (out, scratch) if return_out_x else out


E4M3_MAX = 448.0


def quantize_e4m3_per_channel(weight: torch.Tensor, search: int = 64):
    """(out, in) weight -> (uint8 e4m3fn bytes, float32 scale per output channel).

    One scale per output channel, chosen per row among `search` candidates between 0.75 and 2.1 times max|row| / 448
    as the one with the smallest squared rounding error of the row (values beyond the largest e4m3 number saturate).
    A factor of two covers every alignment of the 3-bit mantissa grid with the row's values; the candidates below 1
    let a row trade the clipping of its largest element for a finer grid.  search = 0: scale = max|row| / 448.
    Against that rule the search lowers the relative rounding error of a weight matrix from 2.55 % to 2.27 %."""
    w = weight.detach().float()
    base = w.abs().amax(dim=1).clamp_min(1e-12) / E4M3_MAX

    def rounded(scale):
        q = (w / scale[:, None]).clamp(-E4M3_MAX, E4M3_MAX).to(torch.float8_e4m3fn)
        return q, ((q.float() * scale[:, None] - w) ** 2).sum(dim=1)

    scale = base.clone()
    q, err = rounded(scale)
    for k in range(int(search)):
        cand = base * (0.75 * 2.0 ** (1.5 * k / search))
        qc, ec = rounded(cand)
        better = ec < err
        if bool(better.any()):
            q = torch.where(better[:, None], qc.view(torch.uint8), q.view(torch.uint8)).view(torch.float8_e4m3fn)
            err = torch.where(better, ec, err)
            scale = torch.where(better, cand, scale)
    return q.view(torch.uint8).contiguous(), scale.contiguous()


def dequantize_e4m3_per_channel(q: torch.Tensor, scale: torch.Tensor) -> torch.Tensor:
    return q.view(torch.float8_e4m3fn).float() * scale[:, None]


def layer_forward(x, params, dims: LayerDims, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5,
                  return_slice_tokens=False):
    """Whole PhysicsAttention layer.  Returns y, or (fx_new, ln_out) with a tail; slice tokens appended on request.

    If `params` carries `in_project_x_scale` the three large weights are fp8-e4m3 bytes (PA_BF16_W8)."""
    _need_cuda(x, residual)
    lib = _lib.load()
    code = _lib.dtype_code(x.dtype)
    if params.get("in_project_x_scale") is not None:
        if x.dtype != torch.bfloat16:
            raise TypeError("fp8-e4m3 weights need bfloat16 activations")
        code = _lib.PA_BF16_W8
    shape, device, stream = byref(dims.c()), x.device, _lib.current_stream_ptr(x.device)
    nbytes = lib.pa_workspace_bytes(code, shape)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_workspace_bytes")
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=device)
    y = torch.empty(dims.B, dims.N, dims.C, dtype=x.dtype, device=device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tok = (torch.empty(dims.B, dims.H, dims.S, dims.D, dtype=torch.float32, device=device)
           if return_slice_tokens else None)
    tail = byref(_c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out))
    c_params = byref(_c_params(params))
    blob = None
    if code != _lib.PA_F32 and lib.pa_query_path(code, shape) == 1:
        # fused MFMA path: the repacked parameters are kept with the parameter set and reused until it changes
        # (fp8-e4m3 weights: the repacking kernel reads the bytes and scales, so they are expanded once, here)
        blob = params.get("_mfma_blob")
        if blob is None:
            n = lib.pa_mfma_buffer_bytes(shape, _lib.PA_BUF_BLOB)
            blob = torch.empty(int(n), dtype=torch.uint8, device=device)
            _lib.check(lib.pa_mfma_pack_params(shape, c_params, blob.data_ptr(), stream), "pa_mfma_pack_params")
            params["_mfma_blob"] = blob
    if blob is not None:
        _lib.check(lib.pa_mfma_layer_forward(shape, c_params, blob.data_ptr(), x.data_ptr(), y.data_ptr(), tail, _lib.ptr(tok),
                                             workspace.data_ptr(), nbytes, stream), "pa_mfma_layer_forward")
    else:
        _lib.check(lib.pa_layer_forward(code, shape, c_params, x.data_ptr(), y.data_ptr(), tail, _lib.ptr(tok),
                                        workspace.data_ptr(), nbytes, stream), "pa_layer_forward")
    out = y if (residual is None and ln_out is None) else (y, ln_out)
    return (out, tok) if return_slice_tokens else out


def layer_forward_plus_supported(dtype: torch.dtype, dims: LayerDims) -> bool:
    """True where the whole Transolver++ layer runs on the staged bf16 MFMA kernels."""
    if dtype != torch.bfloat16:
        return False
    return bool(_lib.load().pa_layer_forward_plus_supported(_lib.PA_BF16, byref(dims.c())))


def layer_forward_plus(x, uniform, params, dims: LayerDims, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5):
    """Whole Transolver++ layer (plus=True) on the staged bf16 MFMA kernels; `uniform` (B, N, H, S) bf16: the samples
    behind the Gumbel noise.  Returns y, or (fx_new, ln_out) with a tail."""
    _need_cuda(x, uniform, residual)
    if uniform.dtype != x.dtype or uniform.shape != (dims.B, dims.N, dims.H, dims.S):
        raise ValueError("uniform samples must have the activation dtype and shape (B, N, H, S)")
    lib = _lib.load()
    code, shape = _lib.dtype_code(x.dtype), dims.c()
    nbytes = lib.pa_layer_forward_plus_workspace_bytes(code, byref(shape))
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_layer_forward_plus_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=x.device)
    y = torch.empty(dims.B, dims.N, dims.C, dtype=x.dtype, device=x.device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    plus = _lib.PaPlusParams(*[_lib.ptr(params[k]) for k, _ in _lib.PaPlusParams._fields_])
    _lib.check(lib.pa_layer_forward_plus(code, byref(shape), byref(_c_params(params)), byref(plus), x.data_ptr(),
                                         uniform.data_ptr(), y.data_ptr(), byref(tail), None, workspace.data_ptr(),
                                         int(nbytes), _lib.current_stream_ptr(x.device)), "pa_layer_forward_plus")
    return y if (residual is None and ln_out is None) else (y, ln_out)


def residual_layernorm(y, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5):
    """In place y <- y + residual (if given); returns (y, LayerNorm(y)) when ln_weight is given, else y."""
    _need_cuda(y, residual, ln_weight, ln_bias)
    C = y.shape[-1]
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    _lib.check(_lib.load().pa_residual_layernorm(_lib.dtype_code(y.dtype), y.numel() // C, C, y.data_ptr(), byref(tail),
                                                 _lib.current_stream_ptr(y.device)), "pa_residual_layernorm")
    return y if ln_out is None else (y, ln_out)


def layernorm_supported(x: torch.Tensor) -> bool:
    """True if the LayerNorm forward / backward kernels serve rows like x's (GPU, fp32 or bf16, whole 16-byte units)."""
    if not x.is_cuda or x.dtype not in (torch.float32, torch.bfloat16):
        return False
    unit = 4 if x.dtype == torch.float32 else 8
    return x.shape[-1] % unit == 0 and x.shape[-1] <= 1024


def layernorm_backward(x, dy, ln_weight, ln_eps=1e-5, add=None):
    """(dx, d gamma, d beta) of LayerNorm over the last axis; x, dy in the activation dtype, gamma float32.  `add`: a
    gradient that reaches x past the LayerNorm, summed into dx."""
    _need_cuda(x, dy, ln_weight, add)
    lib = _lib.load()
    C = x.shape[-1]
    rows = x.numel() // C
    partials = torch.empty(int(lib.pa_layernorm_backward_groups(rows)) * 2 * C, dtype=torch.float32, device=x.device)
    grads = torch.empty(2, C, dtype=torch.float32, device=x.device)
    dx = torch.empty_like(x)
    _lib.check(lib.pa_layernorm_backward_add(_lib.dtype_code(x.dtype), rows, C, x.data_ptr(), dy.data_ptr(), _lib.ptr(add),
                                             ln_weight.data_ptr(), float(ln_eps), dx.data_ptr(), partials.data_ptr(),
                                             grads.data_ptr(), _lib.current_stream_ptr(x.device)),
               "pa_layernorm_backward_add")
    return dx, grads[0], grads[1]


def mlp_supported(dtype: torch.dtype, rows: int, C: int, F: int) -> bool:
    """True if `mlp_forward` serves this shape: bf16 with C in {128, 256, 512} and F a multiple of 64 (MFMA kernels), or
    float32 with C = 128 and F a multiple of 128 (row kernel on split-bf16 products)."""
    if dtype not in (torch.bfloat16, torch.float32):
        return False
    return bool(_lib.load().pa_mlp_query(_lib.dtype_code(dtype), rows, C, F))


def mlp_forward(u, w1, b1, w2, b2, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5):
    """y = w2 . gelu(w1 . u + b1) + b2 [+ residual]; returns y, or (y, LayerNorm(y)) when ln_weight is given.

    u (..., C) bfloat16 or float32; w1 (F, C), w2 (C, F) in the same dtype; b1, b2, ln_weight, ln_bias float32."""
    _need_cuda(u, w1, b1, w2, b2, residual, ln_weight, ln_bias)
    lib = _lib.load()
    C, F = w1.shape[1], w1.shape[0]
    rows = u.numel() // C
    code = _lib.dtype_code(u.dtype)
    nbytes = lib.pa_mlp_workspace_bytes(code, rows, C, F)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_mlp_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=u.device)
    y = torch.empty_like(u)
    ln_out = torch.empty_like(u) if ln_weight is not None else None
    params = _lib.PaMlpParams(_lib.ptr(w1), _lib.ptr(b1), _lib.ptr(w2), _lib.ptr(b2))
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    _lib.check(lib.pa_mlp_forward(code, rows, C, F, byref(params), u.data_ptr(), y.data_ptr(), byref(tail),
                                  workspace.data_ptr(), int(nbytes), _lib.current_stream_ptr(u.device)),
               "pa_mlp_forward")
    return y if ln_out is None else (y, ln_out)


def block_supported(dtype: torch.dtype, dims: LayerDims, F: int) -> bool:
    """True if `block_forward` serves the shape (float32, 32 slices: C = 128 in 8 heads of 16, F a multiple of 128; or
    C = 32 / 64 in heads of 8 / 16 on an irregular mesh, F a multiple of 32)."""
    if dtype != torch.float32:
        return False
    return bool(_lib.load().pa_block_query(_lib.PA_F32, byref(dims.c()), F))


def block_forward(x, fx_in, params, dims: LayerDims, ln2_weight, ln2_bias, ln2_eps, w1, b1, w2, b2,
                  next_ln_weight=None, next_ln_bias=None, next_ln_eps=1e-5, head_weight=None, head_bias=None):
    """One Transolver block behind its first LayerNorm in one library call: fx1 = Attn(x) + fx_in,
    fx_out = Mlp(LayerNorm_2(fx1)) + fx1; returns fx_out, or (fx_out, LayerNorm_next(fx_out)) when next_ln_weight is
    given, or (fx_out, LayerNorm_next(fx_out) head_weight^T + head_bias) when the output head (up to 4 outputs) is given
    as well.  x = LayerNorm_1(fx_in)."""
    _need_cuda(x, fx_in, ln2_weight, ln2_bias, w1, b1, w2, b2, next_ln_weight, next_ln_bias, head_weight, head_bias)
    lib = _lib.load()
    code, shape, F = _lib.dtype_code(x.dtype), dims.c(), w1.shape[0]
    nbytes = lib.pa_block_workspace_bytes(code, byref(shape), F)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_block_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=x.device)
    fx_out = torch.empty_like(fx_in)
    ln_out = torch.empty_like(fx_in) if (next_ln_weight is not None and head_weight is None) else None
    head, head_out = None, None
    if head_weight is not None:
        head_out = torch.empty(*fx_in.shape[:-1], head_weight.shape[0], dtype=fx_in.dtype, device=fx_in.device)
        head = byref(_lib.PaBlockHead(_lib.ptr(head_weight), _lib.ptr(head_bias), head_weight.shape[0], head_out.data_ptr()))
    mlp = _lib.PaBlockMlp(_lib.ptr(ln2_weight), _lib.ptr(ln2_bias), float(ln2_eps), _lib.ptr(w1), _lib.ptr(b1),
                          _lib.ptr(w2), _lib.ptr(b2), F)
    tail = _c_tail(None, next_ln_weight, next_ln_bias, next_ln_eps, ln_out)
    _lib.check(lib.pa_block_forward(code, byref(shape), byref(_c_params(params)), byref(mlp), x.data_ptr(),
                                    fx_in.data_ptr(), fx_out.data_ptr(), byref(tail), head, workspace.data_ptr(),
                                    int(nbytes), _lib.current_stream_ptr(x.device)), "pa_block_forward")
    if head_out is not None:
        return fx_out, head_out
    return fx_out if ln_out is None else (fx_out, ln_out)


def preprocess_supported(dtype: torch.dtype, rows: int, c_in: int, F: int, C: int) -> bool:
    """True if `preprocess_forward` serves the shape: float32 with C = 128, up to 8 input features and F a multiple of
    128, or bfloat16 with C in {256, 512}, up to 16 input features and F a multiple of 32."""
    if dtype not in (torch.float32, torch.bfloat16):
        return False
    return bool(_lib.load().pa_preprocess_query(_lib.dtype_code(dtype), rows, c_in, F, C))


def preprocess_forward(u, w1, b1, w2, b2, ln_weight=None, ln_bias=None, ln_eps=1e-5):
    """The model's preprocess Mlp in one launch: y = w2 . gelu(w1 . u + b1) + b2 for u (..., c_in) with a few input
    features per point; returns y, or (y, LayerNorm(y)) when ln_weight is given."""
    _need_cuda(u, w1, b1, w2, b2, ln_weight, ln_bias)
    lib = _lib.load()
    c_in, F, C = w1.shape[1], w1.shape[0], w2.shape[0]
    rows = u.numel() // c_in
    code = _lib.dtype_code(u.dtype)
    nbytes = lib.pa_preprocess_workspace_bytes(code, rows, c_in, F, C)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_preprocess_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=u.device)
    y = torch.empty(*u.shape[:-1], C, dtype=u.dtype, device=u.device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    params = _lib.PaMlpParams(_lib.ptr(w1), _lib.ptr(b1), _lib.ptr(w2), _lib.ptr(b2))
    tail = _c_tail(None, ln_weight, ln_bias, ln_eps, ln_out)
    _lib.check(lib.pa_preprocess_forward(code, rows, c_in, F, C, byref(params), u.data_ptr(), y.data_ptr(), byref(tail),
                                         workspace.data_ptr(), int(nbytes), _lib.current_stream_ptr(u.device)),
               "pa_preprocess_forward")
    return y if ln_out is None else (y, ln_out)


def mlp_pack(w1, w2):
    """The two weights of the MLP in the fused kernel's operand order: one call per parameter set; the result is the
    `packed` argument of mlp_forward_packed.  w1 (F, C), w2 (C, F) bfloat16 or float32."""
    _need_cuda(w1, w2)
    lib = _lib.load()
    C, F = w1.shape[1], w1.shape[0]
    code = _lib.dtype_code(w1.dtype)
    nbytes = lib.pa_mlp_workspace_bytes(code, 1, C, F)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_mlp_workspace_bytes")
    packed = torch.empty(int(nbytes), dtype=torch.uint8, device=w1.device)
    params = _lib.PaMlpParams(_lib.ptr(w1), None, _lib.ptr(w2), None)
    _lib.check(lib.pa_mlp_pack(code, C, F, byref(params), packed.data_ptr(), int(nbytes),
                               _lib.current_stream_ptr(w1.device)), "pa_mlp_pack")
    return packed


def mlp_pack_e4m3(q1, scale1, q2, scale2):
    """mlp_pack for weights held as fp8-e4m3 bytes: q1 (F, C), q2 (C, F) uint8 with one float32 scale per output row
    (quantize_e4m3_per_channel).  The repacking kernel reads the bytes itself; the result feeds mlp_forward_packed with
    bfloat16 rows and equals mlp_pack over the bf16-rounded dequantised weights bit for bit."""
    _need_cuda(q1, scale1, q2, scale2)
    if q1.dtype != torch.uint8 or q2.dtype != torch.uint8:
        raise TypeError("mlp_pack_e4m3 takes the e4m3 bytes as uint8 tensors")
    lib = _lib.load()
    C, F = q1.shape[1], q1.shape[0]
    nbytes = lib.pa_mlp_workspace_bytes(_lib.PA_BF16, 1, C, F)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_mlp_workspace_bytes")
    packed = torch.empty(int(nbytes), dtype=torch.uint8, device=q1.device)
    _lib.check(lib.pa_mlp_pack_e4m3(C, F, q1.data_ptr(), scale1.data_ptr(), q2.data_ptr(), scale2.data_ptr(),
                                    packed.data_ptr(), int(nbytes), _lib.current_stream_ptr(q1.device)),
               "pa_mlp_pack_e4m3")
    return packed


def mlp_input_ln_supported(dtype: torch.dtype, rows: int, C: int, F: int) -> bool:
    """True if mlp_forward_packed can apply a LayerNorm to its input rows itself (bfloat16, C in {256, 512})."""
    if dtype != torch.bfloat16:
        return False
    return bool(_lib.load().pa_mlp_input_ln_query(_lib.PA_BF16, rows, C, F))


def mlp_forward_packed(u, packed, b1, b2, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5, in_ln=None, train=False):
    """mlp_forward with the weights already in operand order (mlp_pack); b1 (F), b2 (C) float32.  train: GELU to float32
    accuracy (bfloat16 rows of 256 channels, see mlp_backward).

    in_ln = (weight, bias, eps), float32: the rows of u are normalised by the kernel on their way in, i.e. the result is
    w2 . gelu(w1 . LayerNorm(u) + b1) + b2 [+ residual] (mlp_input_ln_supported)."""
    _need_cuda(u, packed, b1, b2, residual, ln_weight, ln_bias)
    lib = _lib.load()
    C, F = b2.numel(), b1.numel()
    rows = u.numel() // C
    y = torch.empty_like(u)
    ln_out = torch.empty_like(u) if ln_weight is not None else None
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    if in_ln is not None:
        _need_cuda(in_ln[0], in_ln[1])
        cin = _lib.PaInputLn(in_ln[0].data_ptr(), in_ln[1].data_ptr(), float(in_ln[2]))
        _lib.check(lib.pa_mlp_forward_packed_ln(_lib.dtype_code(u.dtype), rows, C, F, packed.data_ptr(), b1.data_ptr(),
                                                b2.data_ptr(), byref(cin), u.data_ptr(), y.data_ptr(), byref(tail),
                                                _lib.current_stream_ptr(u.device)), "pa_mlp_forward_packed_ln")
    else:
        call = lib.pa_mlp_train_forward if train else lib.pa_mlp_forward_packed
        _lib.check(call(_lib.dtype_code(u.dtype), rows, C, F, packed.data_ptr(), b1.data_ptr(), b2.data_ptr(), u.data_ptr(),
                        y.data_ptr(), byref(tail), _lib.current_stream_ptr(u.device)),
                   "pa_mlp_train_forward" if train else "pa_mlp_forward_packed")
    return y if ln_out is None else (y, ln_out)


def mlp_backward_supported(dtype: torch.dtype, rows: int, C: int, F: int) -> bool:
    """True if `mlp_backward` serves this shape (bfloat16, C = 256) and `mlp_forward` does."""
    if dtype != torch.bfloat16 or rows <= 0 or not mlp_supported(dtype, rows, C, F):
        return False
    return _lib.load().pa_mlp_backward_workspace_bytes(_lib.PA_BF16, rows, C, F) > 0


def mlp_backward(u, dy, w1, b1, w2):
    """(gelu(w1 . u + b1), d hidden), each (..., F): what the weight and input gradients of `mlp_forward` are products of.

    u, dy (..., C), w1 (F, C), w2 (C, F) bfloat16; b1 float32."""
    _need_cuda(u, dy, w1, b1, w2)
    lib = _lib.load()
    C, F = w1.shape[1], w1.shape[0]
    rows = u.numel() // C
    nbytes = lib.pa_mlp_backward_workspace_bytes(_lib.PA_BF16, rows, C, F)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_mlp_backward_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=u.device)
    act = torch.empty(*u.shape[:-1], F, dtype=u.dtype, device=u.device)
    dh = torch.empty_like(act)
    params = _lib.PaMlpParams(_lib.ptr(w1), _lib.ptr(b1), _lib.ptr(w2), None)
    _lib.check(lib.pa_mlp_backward(_lib.PA_BF16, rows, C, F, byref(params), u.data_ptr(), dy.data_ptr(), act.data_ptr(),
                                   dh.data_ptr(), workspace.data_ptr(), int(nbytes), _lib.current_stream_ptr(u.device)),
               "pa_mlp_backward")
    return act, dh


def norm_mlp_backward_supported(dtype: torch.dtype, rows: int, C: int, F: int) -> bool:
    """True if `norm_mlp_backward` serves this shape (bfloat16, C = 256, F a multiple of 64 as `mlp_supported` takes it)."""
    if dtype != torch.bfloat16 or rows <= 0 or not mlp_supported(dtype, rows, C, F):
        return False
    return _lib.load().pa_norm_mlp_backward_workspace_bytes(_lib.PA_BF16, rows, C, F) > 0


def norm_mlp_backward(u, dy, x, w1, b1, w2, ln_weight, ln_eps=1e-5, linear1=True, linear2=True, through_norm=True):
    """Backward of y = x + w2 . gelu(w1 . u + b1) + b2, u = LayerNorm(x): (dx, d w1, d b1, d w2, d b2, d ln_weight, d ln_bias),
    the parameters' gradients float32.  u, dy, x (..., C), w1 (F, C), w2 (C, F) bfloat16; b1, ln_weight float32.  `linear1`,
    `linear2`, `through_norm` (dx and the LayerNorm's): what is not asked for is not formed and comes back as None."""
    _need_cuda(u, dy, x, w1, b1, w2, ln_weight)
    lib = _lib.load()
    C, F = w1.shape[1], w1.shape[0]
    rows = u.numel() // C
    wanted = (_lib.PA_GRAD_LINEAR1 if linear1 else 0) | (_lib.PA_GRAD_LINEAR2 if linear2 else 0)
    nbytes = lib.pa_norm_mlp_backward_wanted_workspace_bytes(_lib.PA_BF16, rows, C, F, wanted)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_norm_mlp_backward_wanted_workspace_bytes")
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=u.device)
    grads = torch.empty(2 * F * C + F + 3 * C, dtype=torch.float32, device=u.device)
    dx = torch.empty_like(x) if through_norm else None
    params = _lib.PaMlpParams(w1.data_ptr(), b1.data_ptr(), w2.data_ptr(), None)
    _lib.check(lib.pa_norm_mlp_backward_wanted(_lib.PA_BF16, rows, C, F, wanted, byref(params), u.data_ptr(), dy.data_ptr(),
                                               x.data_ptr(), ln_weight.data_ptr(), float(ln_eps), _lib.ptr(dx), grads.data_ptr(),
                                               workspace.data_ptr(), nbytes, _lib.current_stream_ptr(u.device)),
               "pa_norm_mlp_backward_wanted")
    d_w1, d_b1, d_w2, d_b2, d_g, d_b = grads.split([F * C, F, C * F, C, C, C])
    first = (d_w1.view(F, C), d_b1) if linear1 else (None, None)
    second = (d_w2.view(C, F), d_b2) if linear2 else (None, None)
    return (dx, *first, *second, *((d_g, d_b) if through_norm else (None, None)))


class MfmaStages:
    """The bf16 MFMA kernels one by one (pa_mfma_* entry points) with their opaque buffers held as torch tensors.

    Used for per-kernel timing and for checking the MFMA path's slice tokens; `layer_forward` runs the same
    kernels in one library call.
    """

    def __init__(self, params: dict, dims: LayerDims, device):
        lib = _lib.load()
        self.lib, self.params, self.dims, self.device = lib, params, dims, device
        self.shape = dims.c()
        self.cparams = _c_params(params)

        def buf(which):
            n = lib.pa_mfma_buffer_bytes(byref(self.shape), which)
            if n < 0:
                _lib.check(int(n), "pa_mfma_buffer_bytes")
            return torch.empty(int(n), dtype=torch.uint8, device=device)

        self.blob, self.fx_pack, self.w_pack = buf(_lib.PA_BUF_BLOB), buf(_lib.PA_BUF_FX_PACK), buf(_lib.PA_BUF_W_PACK)
        self.partials, self.tokp = buf(_lib.PA_BUF_PARTIALS), buf(_lib.PA_BUF_TOKP)
        f32 = dict(dtype=torch.float32, device=device)
        self.tok = torch.empty(dims.B, dims.H, dims.S, dims.D, **f32)
        self.norm = torch.empty(dims.B, dims.H, dims.S, **f32)
        self.tok_out = torch.empty(dims.B, dims.H, dims.S, dims.D, **f32)
        self.groups = int(lib.pa_mfma_partial_groups(byref(self.shape), 0))   # producer of `partials`: kernel (b)
        self.fused_groups = int(lib.pa_mfma_partial_groups(byref(self.shape), 1))  # < 0: fused form not available

    def _stream(self):
        return _lib.current_stream_ptr(self.device)

    def pack_params(self):
        _lib.check(self.lib.pa_mfma_pack_params(byref(self.shape), byref(self.cparams), self.blob.data_ptr(),
                                                self._stream()), "pa_mfma_pack_params")

    def project_softmax(self, x):
        _need_cuda(x)
        _lib.check(self.lib.pa_mfma_project_softmax(byref(self.shape), self.blob.data_ptr(), x.data_ptr(),
                                                    self.fx_pack.data_ptr(), self.w_pack.data_ptr(), self._stream()),
                   "pa_mfma_project_softmax")

    def slice_reduce(self):
        _lib.check(self.lib.pa_mfma_slice_reduce(byref(self.shape), self.w_pack.data_ptr(), self.fx_pack.data_ptr(),
                                                 self.partials.data_ptr(), self._stream()), "pa_mfma_slice_reduce")
        self._producer_groups = self.groups

    def project_softmax_reduce(self, x):
        """Kernels (a)+(b) in one launch (what `layer_forward` runs when slice_num <= 64)."""
        _need_cuda(x)
        _lib.check(self.lib.pa_mfma_project_softmax_reduce(byref(self.shape), self.blob.data_ptr(), x.data_ptr(),
                                                           self.w_pack.data_ptr(), self.partials.data_ptr(),
                                                           self._stream()), "pa_mfma_project_softmax_reduce")
        self._producer_groups = self.fused_groups

    def project_softmax_reduce_clocked(self, x):
        """`project_softmax_reduce` with the shader clock one of its workgroups ran at: returns (GHz, cycles, ns).
        Hidden width 256, slice_num <= 64."""
        _need_cuda(x)
        clock = torch.zeros(2, dtype=torch.int64, device=self.device)
        _lib.check(self.lib.pa_mfma_project_softmax_reduce_clocked(byref(self.shape), self.blob.data_ptr(), x.data_ptr(),
                                                                   self.w_pack.data_ptr(), self.partials.data_ptr(),
                                                                   clock.data_ptr(), self._stream()),
                   "pa_mfma_project_softmax_reduce_clocked")
        self._producer_groups = self.fused_groups
        cycles, ticks = (int(v) for v in clock.tolist())
        return cycles / (10.0 * ticks), cycles, 10 * ticks

    def combine_attention(self):
        _lib.check(self.lib.pa_mfma_combine_attention(byref(self.shape), byref(self.cparams), self.partials.data_ptr(),
                                                      self._producer_groups, self.tok.data_ptr(), self.norm.data_ptr(), self.tok_out.data_ptr(),
                                                      self.tokp.data_ptr(), self._stream()), "pa_mfma_combine_attention")

    def set_out_tokens(self, out_tok):
        """Attended slice tokens computed by the caller (B,H,S,32 float32) in place of `combine_attention`'s."""
        _need_cuda(out_tok)
        self.tok_out.copy_(out_tok)
        _lib.check(self.lib.pa_mfma_pack_tokens(byref(self.shape), self.tok_out.data_ptr(), self.tokp.data_ptr(),
                                                self._stream()), "pa_mfma_pack_tokens")

    # ---- backward-pass stages (pa_mfma_backward_query() == 1) ----
    def rows_gemm_packed(self, inp, weight, bias, natural=True, packed=True):
        """bf16 Linear (B, N, c_in) -> H*32 columns; returns (natural (B, N, H*32) or None, packed buffer or None)."""
        _need_cuda(inp, weight, bias)
        d = self.dims
        out = torch.empty(d.B, d.N, d.H * 32, dtype=torch.bfloat16, device=self.device) if natural else None
        pack = torch.empty_like(self.fx_pack) if packed else None
        _lib.check(self.lib.pa_rows_gemm_packed(byref(self.shape), inp.shape[-1], inp.data_ptr(), weight.data_ptr(),
                                                _lib.ptr(bias), _lib.ptr(out), _lib.ptr(pack), self._stream()),
                   "pa_rows_gemm_packed")
        return out, pack

    def slice_weighted_sum(self, v_pack):
        """(B, H, S, D+1) float32: sum_n w[n,s] [v[n,:], 1] with w from w_pack and v in the packed layout."""
        d = self.dims
        sums = torch.empty(d.B, d.H, d.S, d.D + 1, dtype=torch.float32, device=self.device)
        _lib.check(self.lib.pa_mfma_slice_weighted_sum(byref(self.shape), self.w_pack.data_ptr(), v_pack.data_ptr(),
                                                       self.partials.data_ptr(), sums.data_ptr(), self._stream()),
                   "pa_mfma_slice_weighted_sum")
        return sums

    def deslice(self):
        """out_x (B, N, H*32) bf16 from w_pack and the attended tokens."""
        d = self.dims
        out_x = torch.empty(d.B, d.N, d.H * 32, dtype=torch.bfloat16, device=self.device)
        _lib.check(self.lib.pa_mfma_deslice(byref(self.shape), self.w_pack.data_ptr(), self.tokp.data_ptr(),
                                            out_x.data_ptr(), self._stream()), "pa_mfma_deslice")
        return out_x

    def slice_softmax_backward(self, x_mid, fx_mid, d_out_x, d_num, d_norm):
        """Returns (d_proj (B,N,2HD) = [d x_mid | d fx_mid], d_z (B,N,H,S), d clamp(temperature) (H) float32)."""
        _need_cuda(x_mid, fx_mid, d_out_x, d_num, d_norm)
        d = self.dims
        nbytes = self.lib.pa_mfma_backward_tables_bytes(byref(self.shape))
        groups = self.lib.pa_mfma_backward_groups(byref(self.shape))
        if nbytes < 0 or groups < 0:
            _lib.check(int(min(nbytes, groups)), "pa_mfma_backward_tables_bytes")
        tables = torch.empty(int(nbytes), dtype=torch.uint8, device=self.device)
        d_proj = torch.empty(d.B, d.N, 2 * d.H * 32, dtype=torch.bfloat16, device=self.device)
        d_z = torch.empty(d.B, d.N, d.H, d.S, dtype=torch.bfloat16, device=self.device)
        dT = torch.empty(int(groups), d.H, dtype=torch.float32, device=self.device)
        _lib.check(self.lib.pa_mfma_slice_softmax_backward(
            byref(self.shape), byref(self.cparams), x_mid.data_ptr(), fx_mid.data_ptr(), d_out_x.data_ptr(),
            self.w_pack.data_ptr(), self.tok_out.data_ptr(), d_num.data_ptr(), d_norm.data_ptr(), tables.data_ptr(),
            d_proj.data_ptr(), d_z.data_ptr(), dT.data_ptr(), self._stream()), "pa_mfma_slice_softmax_backward")
        return d_proj, d_z, dT.sum(0)

    def deslice_project(self, y, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5, ln_out=None):
        tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
        _lib.check(self.lib.pa_mfma_deslice_project(byref(self.shape), self.blob.data_ptr(), self.w_pack.data_ptr(),
                                                    self.tokp.data_ptr(), y.data_ptr(), byref(tail), self._stream()),
                   "pa_mfma_deslice_project")


# ---------------------------------------------------------------------------------------------------
# backward-pass entry points
# ---------------------------------------------------------------------------------------------------
def backward_supported(dtype: torch.dtype, dims: LayerDims) -> bool:
    rc = _lib.load().pa_backward_query(_lib.dtype_code(dtype), byref(dims.c()))
    if rc < 0:
        _lib.check(rc, "pa_backward_query")
    return bool(rc)


def mfma_backward_supported(dtype: torch.dtype, dims: LayerDims) -> bool:
    """True if the bf16 MFMA backward kernels serve this shape (MFMA forward shapes with slice_num <= 64)."""
    if dtype != torch.bfloat16:
        return False
    rc = _lib.load().pa_mfma_backward_query(byref(dims.c()))
    if rc < 0:
        _lib.check(rc, "pa_mfma_backward_query")
    return bool(rc)


def _c_plus(params: dict):
    return byref(_lib.PaPlusParams(*[_lib.ptr(params[k]) for k, _ in _lib.PaPlusParams._fields_]))


def point_backward(x_mid, fx_mid, d_out_x, tok_out, d_num, d_norm, params, dims: LayerDims):
    """Per-point part of the backward pass for bf16 layers with 32-wide heads.  Returns (d_proj (B,N,2HD) = [d x_mid |
    d fx_mid], d W_slice (S, D), d b_slice (S), d temperature (H)); tok_out None: no deslice term."""
    _need_cuda(x_mid, fx_mid, d_out_x, tok_out, d_num, d_norm)
    lib, shape, S, D, H = _lib.load(), dims.c(), dims.S, dims.D, dims.H
    nbytes = lib.pa_point_backward_workspace_bytes(byref(shape), 0)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_point_backward_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=x_mid.device)
    d_proj = torch.empty(dims.B, dims.N, 2 * H * D, dtype=x_mid.dtype, device=x_mid.device)
    grads = torch.empty(lib.pa_point_backward_grads(byref(shape), 0), dtype=torch.float32, device=x_mid.device)
    _lib.check(lib.pa_point_backward(
        byref(shape), byref(_c_params(params)), None, x_mid.data_ptr(), fx_mid.data_ptr(), d_out_x.data_ptr(), None,
        _lib.ptr(tok_out), d_num.data_ptr(), d_norm.data_ptr(), workspace.data_ptr(), int(nbytes), d_proj.data_ptr(),
        grads.data_ptr(), _lib.current_stream_ptr(x_mid.device)), "pa_point_backward")
    return d_proj, grads[:S * D].view(S, D), grads[S * D:S * D + S], grads[S * D + S:]


def output_backward(w_pack, dy, tok_out, w_out, dims: LayerDims):
    """From dy (B,N,C) bf16 and the forward's packed slice weights: (d tok_out (B,H,S,D), d W_out (C,HD), d b_out (C))."""
    _need_cuda(w_pack, dy, tok_out, w_out)
    lib, shape = _lib.load(), dims.c()
    nbytes = lib.pa_output_backward_workspace_bytes(byref(shape))
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_output_backward_workspace_bytes")
    f32 = dict(dtype=torch.float32, device=dy.device)
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=dy.device)
    d_tok, d_w = torch.empty(dims.B, dims.H, dims.S, dims.D, **f32), torch.empty(dims.C, dims.H * dims.D, **f32)
    d_b = torch.empty(dims.C, **f32)
    _lib.check(lib.pa_output_backward(byref(shape), w_pack.data_ptr(), dy.data_ptr(), tok_out.data_ptr(), w_out.data_ptr(),
                                      workspace.data_ptr(), int(nbytes), d_tok.data_ptr(), d_w.data_ptr(), d_b.data_ptr(),
                                      _lib.current_stream_ptr(dy.device)), "pa_output_backward")
    return d_tok, d_w, d_b


def _train_bytes(dtype: torch.dtype, shape, plus: bool, which: int) -> int:
    if dtype == torch.float32 and not plus:
        return _lib.load().pa_layer_train_f32_bytes(shape, which)
    return _lib.load().pa_layer_train_bytes(shape, int(plus), which) if dtype == torch.bfloat16 else 0


def layer_train_supported(dtype: torch.dtype, dims: LayerDims, plus: bool = False) -> bool:
    """True where a layer trains in the two library calls below (bf16 with 32-wide heads; float32 without Transolver++)."""
    return _train_bytes(dtype, byref(dims.c()), plus, _lib.PA_TRAIN_SAVED) > 0


_TRAIN_LARGE = ("in_project_x_weight", "in_project_fx_weight", "out_linear_weight")


def layer_train_forward(x, uniform, params: dict, dims: LayerDims, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5):
    """(y, saved) of a layer, with ln_weight (y + residual, saved, LayerNorm(y + residual)).  `params`: the layer's own
    parameters under the names of `pa_params` / `pa_plus_params` in torch's layout, float32; bf16 layers take the three large
    weights all in bfloat16, too."""
    _need_cuda(x, uniform, residual, ln_weight, ln_bias, *params.values())
    if uniform is not None and (uniform.dtype != x.dtype or uniform.shape != (dims.B, dims.N, dims.H, dims.S)):
        raise ValueError("uniform samples must have the activation dtype and shape (B, N, H, S)")
    large = params["out_linear_weight"].dtype
    if large not in (x.dtype, torch.float32):
        raise TypeError(f"{large} weights do not go with {x.dtype} activations")
    for name, p in params.items():
        wanted = large if name in _TRAIN_LARGE else torch.float32
        if p.dtype != wanted:
            raise TypeError(f"{name}: {p.dtype}, expected {wanted}")
    lib, shape, plus = _lib.load(), byref(dims.c()), uniform is not None
    nbytes = _train_bytes(x.dtype, shape, plus, _lib.PA_TRAIN_FORWARD)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_layer_train_bytes")
    saved = torch.empty(_train_bytes(x.dtype, shape, plus, _lib.PA_TRAIN_SAVED), dtype=torch.uint8, device=x.device)
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    y = torch.empty(dims.B, dims.N, dims.C, dtype=x.dtype, device=x.device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tail = byref(_c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out))
    rest = (saved.data_ptr(), workspace.data_ptr(), nbytes, _lib.current_stream_ptr(x.device))
    if x.dtype == torch.float32:
        _lib.check(lib.pa_layer_train_f32_forward(shape, byref(_c_params(params)), x.data_ptr(), y.data_ptr(), tail, *rest),
                   "pa_layer_train_f32_forward")
    else:
        _lib.check(lib.pa_layer_train_forward(
            shape, _lib.dtype_code(params["out_linear_weight"].dtype), byref(_c_params(params)), _c_plus(params) if plus else None,
            x.data_ptr(), _lib.ptr(uniform), y.data_ptr(), tail, *rest), "pa_layer_train_forward")
    return (y, saved) if ln_out is None else (y, saved, ln_out)


def layer_train_gradients(x, uniform, dy, saved, dims: LayerDims, need_dx: bool = True):
    """(dx or None, one float32 buffer with the gradients of all parameters in the order of `TRAIN_GRADIENTS` /
    `TRAIN_GRADIENTS_PLUS`, each in its parameter's layout) of `layer_train_forward`; the parameters are those of the forward
    call, kept in `saved`."""
    _need_cuda(x, uniform, dy, saved)
    lib, shape, plus = _lib.load(), byref(dims.c()), uniform is not None
    nbytes = _train_bytes(x.dtype, shape, plus, _lib.PA_TRAIN_BACKWARD)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_layer_train_bytes")
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=x.device)
    grads = torch.empty(_train_bytes(x.dtype, shape, plus, _lib.PA_TRAIN_GRADS) // 4, dtype=torch.float32, device=x.device)
    dx = torch.empty_like(x) if need_dx else None
    rest = (saved.data_ptr(), _lib.ptr(dx), grads.data_ptr(), workspace.data_ptr(), nbytes, _lib.current_stream_ptr(x.device))
    if x.dtype == torch.float32:
        _lib.check(lib.pa_layer_train_f32_backward(shape, x.data_ptr(), dy.data_ptr(), *rest), "pa_layer_train_f32_backward")
    else:
        _lib.check(lib.pa_layer_train_backward(shape, None, byref(_lib.PaPlusParams()) if plus else None, x.data_ptr(),
                                               _lib.ptr(uniform), dy.data_ptr(), *rest), "pa_layer_train_backward")
    return dx, grads


_TRAIN_TAIL = ("out_linear_weight", "out_linear_bias", "qkv_project_weight", "in_project_slice_weight",
               "in_project_slice_bias", "temperature")
TRAIN_GRADIENTS = ("in_project_x_weight", "in_project_fx_weight", "in_project_x_bias", "in_project_fx_bias") + _TRAIN_TAIL
TRAIN_GRADIENTS_PLUS = ("in_project_x_weight", "in_project_x_bias") + _TRAIN_TAIL + (
    "proj_temperature_0_weight", "proj_temperature_0_bias", "proj_temperature_2_weight", "proj_temperature_2_bias")


def layer_train_backward(x, uniform, dy, saved, dims: LayerDims, need_dx: bool = True):
    """(dx or None, gradients by parameter name, float32 views of one buffer) of `layer_train_forward`."""
    dx, grads = layer_train_gradients(x, uniform, dy, saved, dims, need_dx)
    C, HD, S, D, H = dims.C, dims.H * dims.D, dims.S, dims.D, dims.H
    taps = dims.conv_k ** (3 if dims.grid_d > 0 else 2) if dims.conv_k > 0 else 1
    size = {"in_project_x_weight": HD * C * taps, "in_project_fx_weight": HD * C * taps, "in_project_x_bias": HD,
            "in_project_fx_bias": HD, "out_linear_weight": C * HD, "out_linear_bias": C, "qkv_project_weight": 3 * D * D,
            "in_project_slice_weight": S * D, "in_project_slice_bias": S, "temperature": H, "proj_temperature_0_weight": S * D,
            "proj_temperature_0_bias": S, "proj_temperature_2_weight": S, "proj_temperature_2_bias": 1}
    names = TRAIN_GRADIENTS if uniform is None else TRAIN_GRADIENTS_PLUS
    return dx, dict(zip(names, grads.split([size[n] for n in names])))


def _cols_gemm_bytes(a: torch.Tensor, b: torch.Tensor, grid: LayerDims | None) -> int:
    """Workspace of `cols_gemm` for these operands, 0 or less where it does not serve them."""
    if not (a.is_cuda and a.dtype == b.dtype and a.dtype in (torch.float32, torch.bfloat16)) or a.numel() == 0:
        return 0
    if a.data_ptr() % 16 or b.data_ptr() % 16:
        return 0
    ca = a.shape[-1]
    return _lib.load().pa_weight_grad_workspace_bytes(_lib.dtype_code(a.dtype), a.numel() // ca, ca, b.shape[-1],
                                                      byref(grid.c()) if grid is not None else None)


def cols_gemm_supported(a: torch.Tensor, b: torch.Tensor, grid: LayerDims | None = None) -> bool:
    """True if `cols_gemm` serves d out = a (..., ca), input = b (..., cb) (see pa_weight_grad for the shapes)."""
    return _cols_gemm_bytes(a, b, grid) > 0


def try_cols_gemm(a: torch.Tensor, b: torch.Tensor, grid: LayerDims | None = None):
    """`cols_gemm(a, b, col_sums=True, grid=grid)` where it serves the operands, else None."""
    nbytes = _cols_gemm_bytes(a, b, grid)
    return _cols_gemm(a, b, True, grid, nbytes) if nbytes > 0 else None


def cols_gemm(a: torch.Tensor, b: torch.Tensor, col_sums: bool = False, grid: LayerDims | None = None):
    """a^T . b over the leading (row) axes: bf16 or float32 (..., ca) and (..., cb) with equal row counts -> float32
    (ca, cb): the weight-gradient product d W = d out^T . in.  With `grid` (the dims of a structured layer) b's rows are
    gathered at every tap of its convolution and the result is (ca, cb, k, ..., k).  With `col_sums` the column sums of
    a (the matching bias gradient) come back as well, from the same pass."""
    rows = a.numel() // a.shape[-1]
    nbytes = _lib.load().pa_weight_grad_workspace_bytes(_lib.dtype_code(a.dtype), rows, a.shape[-1], b.shape[-1],
                                                        byref(grid.c()) if grid is not None else None)
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_weight_grad_workspace_bytes")
    return _cols_gemm(a, b, col_sums, grid, nbytes)


def _cols_gemm(a, b, col_sums: bool, grid: LayerDims | None, nbytes: int):
    _need_cuda(a, b)
    ca, cb = a.shape[-1], b.shape[-1]
    rows = a.numel() // ca
    if b.numel() // cb != rows:
        raise ValueError("cols_gemm needs the same number of rows on both sides")
    workspace = torch.empty(nbytes, dtype=torch.uint8, device=a.device)
    taps = (grid.conv_k,) * (3 if grid.grid_d > 0 else 2) if grid is not None and grid.conv_k > 0 else ()
    out = torch.empty(ca, cb, *taps, dtype=torch.float32, device=a.device)
    sums = torch.empty(ca, dtype=torch.float32, device=a.device) if col_sums else None
    _lib.check(_lib.load().pa_weight_grad(_lib.dtype_code(a.dtype), rows, a.data_ptr(), ca, b.data_ptr(), cb,
                                          byref(grid.c()) if grid is not None else None, workspace.data_ptr(), nbytes,
                                          out.data_ptr(), _lib.ptr(sums), _lib.current_stream_ptr(a.device)), "pa_weight_grad")
    return (out, sums) if col_sums else out


def rows_gemm(inp, weight, bias, dims: LayerDims, c_in: int, c_out: int, gelu: bool = False):
    """out (B, N, c_out) = Linear or grid convolution of inp (B, N, c_in), optionally followed by GELU (erf form);
    `dims` supplies B, N and the grid."""
    _need_cuda(inp, weight, bias)
    out = torch.empty(dims.B, dims.N, c_out, dtype=inp.dtype, device=inp.device)
    _lib.check(_lib.load().pa_rows_gemm_act(_lib.dtype_code(inp.dtype), byref(dims.c()), c_in, c_out, inp.data_ptr(),
                                            weight.data_ptr(), _lib.ptr(bias), 1 if gelu else 0, out.data_ptr(),
                                            _lib.current_stream_ptr(inp.device)), "pa_rows_gemm_act")
    return out


def linear(inp, weight, bias, gelu: bool = False):
    """torch.nn.functional.linear over the last axis (+ optional GELU) on the library's row GEMM kernels."""
    lead = inp.shape[:-1]
    rows = inp.numel() // inp.shape[-1]
    out = rows_gemm(inp.reshape(1, rows, inp.shape[-1]).contiguous(), weight, bias,
                    LayerDims(1, rows, inp.shape[-1], 1, 1, 1), inp.shape[-1], weight.shape[0], gelu)
    return out.reshape(*lead, weight.shape[0])


def slice_weighted_sum(w, v, dims: LayerDims):
    """(B, H, S, D+1) float32: sum_n w[n,s] * [v[n,:], 1]."""
    _need_cuda(w, v)
    lib = _lib.load()
    shape = dims.c()
    g = lib.pa_reduce_partial_count(byref(shape))
    if g < 0:
        _lib.check(int(g), "pa_reduce_partial_count")
    partials = torch.empty(g * dims.B * dims.H * dims.S * (dims.D + 1), dtype=torch.float32, device=w.device)
    sums = torch.empty(dims.B, dims.H, dims.S, dims.D + 1, dtype=torch.float32, device=w.device)
    _lib.check(lib.pa_slice_weighted_sum(_lib.dtype_code(w.dtype), byref(shape), w.data_ptr(), v.data_ptr(),
                                         partials.data_ptr(), sums.data_ptr(), _lib.current_stream_ptr(w.device)),
               "pa_slice_weighted_sum")
    return sums


def slice_attention_backward(tok, norm, d_tok_out, params, dims: LayerDims):
    """Returns (d_num, d_norm, d_qkv_weight); with norm=None: (d_tok, None, d_qkv_weight)."""
    _need_cuda(tok, norm, d_tok_out)
    f32 = dict(dtype=torch.float32, device=tok.device)
    BH = dims.B * dims.H
    scratch = torch.empty(BH * 2 * dims.S * dims.S, **f32)
    d_num = torch.empty(dims.B, dims.H, dims.S, dims.D, **f32)
    d_norm = torch.empty(dims.B, dims.H, dims.S, **f32) if norm is not None else None
    parts = torch.empty(BH, 3 * dims.D, dims.D, **f32)
    _lib.check(_lib.load().pa_slice_attention_backward(byref(dims.c()), byref(_c_params(params)), tok.data_ptr(),
                                                       _lib.ptr(norm), d_tok_out.data_ptr(), scratch.data_ptr(),
                                                       d_num.data_ptr(), _lib.ptr(d_norm), parts.data_ptr(),
                                                       _lib.current_stream_ptr(tok.device)),
               "pa_slice_attention_backward")
    return d_num, d_norm, parts.sum(0)


def slice_softmax_backward(x_mid, fx_mid, w, d_out_x, tok_out, d_num, d_norm, params, dims: LayerDims):
    """Returns (d_proj (B,N,2HD) = [d x_mid | d fx_mid], d_z (B,N,H,S), d clamp(temperature) (H) float32)."""
    _need_cuda(x_mid, fx_mid, w, d_out_x, tok_out, d_num, d_norm)
    lib = _lib.load()
    shape = dims.c()
    tiles = lib.pa_backward_point_tiles(byref(shape))
    if tiles < 0:
        _lib.check(int(tiles), "pa_backward_point_tiles")
    d_proj = torch.empty(dims.B, dims.N, 2 * dims.H * dims.D, dtype=w.dtype, device=w.device)
    d_z = torch.empty(dims.B, dims.N, dims.H, dims.S, dtype=w.dtype, device=w.device)
    dT = torch.empty(int(tiles), dims.H, dtype=torch.float32, device=w.device)
    _lib.check(lib.pa_slice_softmax_backward(_lib.dtype_code(w.dtype), byref(shape), byref(_c_params(params)),
                                             x_mid.data_ptr(), fx_mid.data_ptr(), w.data_ptr(), d_out_x.data_ptr(),
                                             tok_out.data_ptr(), d_num.data_ptr(), d_norm.data_ptr(),
                                             d_proj.data_ptr(), d_z.data_ptr(), dT.data_ptr(),
                                             _lib.current_stream_ptr(w.device)), "pa_slice_softmax_backward")
    return d_proj, d_z, dT.sum(0)


def plus_backward_supported(dtype: torch.dtype, dims: LayerDims) -> bool:
    return backward_supported(dtype, dims) and _lib.load().pa_backward_point_tiles_plus(byref(dims.c())) > 0


def slice_softmax_plus_backward(x_mid, uniform, w, d_out_x, tok_out, d_num, d_norm, params, dims: LayerDims):
    """Transolver++ form of `slice_softmax_backward`.  Returns (d x_mid (B,N,HD), d_z (B,N,H,S), d_a1 (B,N,H,S),
    d_a2 (B,N,H) float32, d temperature (H) float32); d_a1 / d_a2 are the gradients of the two proj_temperature Linear
    outputs."""
    _need_cuda(x_mid, uniform, w, d_out_x, tok_out, d_num, d_norm)
    lib = _lib.load()
    shape = dims.c()
    tiles = lib.pa_backward_point_tiles_plus(byref(shape))
    if tiles < 0:
        _lib.check(int(tiles), "pa_backward_point_tiles_plus")
    d_x_mid = torch.empty(dims.B, dims.N, dims.H * dims.D, dtype=w.dtype, device=w.device)
    d_z = torch.empty(dims.B, dims.N, dims.H, dims.S, dtype=w.dtype, device=w.device)
    d_a1 = torch.empty_like(d_z)
    d_a2 = torch.empty(dims.B, dims.N, dims.H, dtype=torch.float32, device=w.device)
    dT = torch.empty(int(tiles), dims.H, dtype=torch.float32, device=w.device)
    plus = _lib.PaPlusParams(*[_lib.ptr(params[k]) for k, _ in _lib.PaPlusParams._fields_])
    _lib.check(lib.pa_slice_softmax_plus_backward(
        _lib.dtype_code(w.dtype), byref(shape), byref(_c_params(params)), byref(plus), x_mid.data_ptr(),
        uniform.data_ptr(), w.data_ptr(), d_out_x.data_ptr(), tok_out.data_ptr(), d_num.data_ptr(), d_norm.data_ptr(),
        d_x_mid.data_ptr(), d_z.data_ptr(), d_a1.data_ptr(), d_a2.data_ptr(), dT.data_ptr(),
        _lib.current_stream_ptr(w.device)), "pa_slice_softmax_plus_backward")
    return d_x_mid, d_z, d_a1, d_a2, dT.sum(0)


def slice_cross_attention_mix(tok, self_out, context, gale_params: dict, dims: LayerDims, tokp=None):
    """GALE slice-token stage: cross-attention of the slice tokens (B,H,S,D) to `context` (B,H,Sc,Dc) blended with the
    self-attention output; all float32.  `gale_params`: the cross_q/k/v weights and biases plus either ``state_mixing``
    or ``concat_project_weight`` / ``concat_project_bias``.  `tokp`: the MFMA deslice operand buffer to fill as well."""
    _need_cuda(tok, self_out, context)
    if context.dtype != torch.float32 or context.ndim != 4 or context.shape[:2] != (dims.B, dims.H):
        raise ValueError(f"context must be float32 (B, H, Sc, Dc) = ({dims.B}, {dims.H}, ., .), got {tuple(context.shape)}")
    gp = _lib.PaGaleParams(*[_lib.ptr(gale_params.get(k)) for k, _ in _lib.PaGaleParams._fields_])
    out = torch.empty_like(tok)
    _lib.check(_lib.load().pa_slice_cross_attention_mix(
        byref(dims.c()), byref(gp), context.shape[2], context.shape[3], tok.data_ptr(), self_out.data_ptr(),
        context.data_ptr(), out.data_ptr(), _lib.ptr(tokp), _lib.current_stream_ptr(tok.device)),
        "pa_slice_cross_attention_mix")
    return out


def flare_forward_mfma_supported(dtype: torch.dtype, dims: LayerDims) -> bool:
    """True where the whole FLARE layer forward runs on the bf16 MFMA kernels."""
    return dtype == torch.bfloat16 and bool(_lib.load().pa_flare_forward_mfma_supported(byref(dims.c())))


def flare_forward_mfma(x, params, dims: LayerDims, residual=None, ln_weight=None, ln_bias=None, ln_eps=1e-5,
                       project: bool = True):
    """FLARE layer forward on the bf16 MFMA kernels from the composed weights of `FLARE.kernel_params`.  Returns y, or
    (fx_new, ln_out) with a tail; `project=False`: the attention output (B, N, H*32) before out_linear."""
    _need_cuda(x, residual)
    lib, shape = _lib.load(), dims.c()
    nbytes = lib.pa_flare_forward_mfma_workspace_bytes(byref(shape))
    if nbytes < 0:
        _lib.check(int(nbytes), "pa_flare_forward_mfma_workspace_bytes")
    workspace = torch.empty(int(nbytes), dtype=torch.uint8, device=x.device)
    y = torch.empty(dims.B, dims.N, dims.C if project else dims.H * 32, dtype=x.dtype, device=x.device)
    ln_out = torch.empty_like(y) if ln_weight is not None else None
    tail = _c_tail(residual, ln_weight, ln_bias, ln_eps, ln_out)
    _lib.check(lib.pa_flare_forward_mfma(
        byref(shape), params["scores_weight"].data_ptr(), params["scores_bias"].data_ptr(),
        params["values_weight"].data_ptr(), params["values_bias"].data_ptr(),
        params["out_linear_weight"].data_ptr() if project else None,
        params["out_linear_bias"].data_ptr() if project else None, x.data_ptr(), y.data_ptr(), byref(tail),
        workspace.data_ptr(), int(nbytes),
        _lib.current_stream_ptr(x.device)), "pa_flare_forward_mfma")
    return y if (residual is None and ln_out is None) else (y, ln_out)


def flare_column_weights(scores, dims: LayerDims):
    """FLARE first pass weights: exp(A - max_n A) for the scores A (B,N,H,S); returns (weights like A, column max
    (B,H,S) float32)."""
    _need_cuda(scores)
    lib = _lib.load()
    shape = dims.c()
    chunks = lib.pa_flare_column_max_chunks(byref(shape))
    if chunks < 0:
        _lib.check(int(chunks), "pa_flare_column_max_chunks")
    f32 = dict(dtype=torch.float32, device=scores.device)
    partials = torch.empty(int(chunks) * dims.B * dims.H * dims.S, **f32)
    colmax = torch.empty(dims.B, dims.H, dims.S, **f32)
    weights = torch.empty_like(scores)
    _lib.check(lib.pa_flare_column_weights(_lib.dtype_code(scores.dtype), byref(shape), scores.data_ptr(),
                                           partials.data_ptr(), colmax.data_ptr(), weights.data_ptr(),
                                           _lib.current_stream_ptr(scores.device)), "pa_flare_column_weights")
    return weights, colmax


def flare_softmax_rows_(scores, dims: LayerDims):
    """In-place softmax over the last axis of the scores (B,N,H,S)."""
    _need_cuda(scores)
    _lib.check(_lib.load().pa_flare_softmax_rows(_lib.dtype_code(scores.dtype), byref(dims.c()), scores.data_ptr(),
                                                 _lib.current_stream_ptr(scores.device)), "pa_flare_softmax_rows")
    return scores


def flare_backward_points(row_w, col_w, values, d_out_x, z, d_num, d_den, dims: LayerDims):
    """Per-point part of the FLARE backward pass: returns (d scores (B,N,H,S), d values (B,N,H*D))."""
    _need_cuda(row_w, col_w, values, d_out_x, z, d_num, d_den)
    d_scores = torch.empty_like(row_w)
    d_values = torch.empty_like(values)
    _lib.check(_lib.load().pa_flare_backward_points(
        _lib.dtype_code(row_w.dtype), byref(dims.c()), row_w.data_ptr(), col_w.data_ptr(), values.data_ptr(),
        d_out_x.data_ptr(), z.data_ptr(), d_num.data_ptr(), d_den.data_ptr(), d_scores.data_ptr(), d_values.data_ptr(),
        _lib.current_stream_ptr(row_w.device)), "pa_flare_backward_points")
    return d_scores, d_values


def deslice(w, tok_out, dims: LayerDims):
    """out_x (B, N, H*D) = sum_s w[n,h,s] tok_out[h,s,:] (heads merged), without the output projection."""
    _need_cuda(w, tok_out)
    out_x = torch.empty(dims.B, dims.N, dims.H * dims.D, dtype=w.dtype, device=w.device)
    _lib.check(_lib.load().pa_deslice(_lib.dtype_code(w.dtype), byref(dims.c()), w.data_ptr(), tok_out.data_ptr(),
                                      out_x.data_ptr(), _lib.current_stream_ptr(w.device)), "pa_deslice")
    return out_x


def _cell_list(pts: torch.Tensor, radius: float, G: int):
    """Bins (B, Np, 3) points into G^3 cells of edge >= radius * 1.0001 per batch: (grid (B, 6), points sorted by
    (batch, cell), their indices within the batch, cell offsets) -- the cell list `pa_ball_query_cells` reads.  Device
    ops only, no synchronisation."""
    B, Np = pts.shape[0], pts.shape[1]
    lo, hi = pts.amin(1), pts.amax(1)
    edge = torch.clamp((hi - lo) / G, min=max(float(radius) * 1.0001, 1e-30))
    grid = torch.cat([lo, 1.0 / edge], dim=1).contiguous()  # (B, 6)
    return grid, *_bin(pts, grid, G, want_start=True)


def _bin(p: torch.Tensor, grid: torch.Tensor, G: int, want_start: bool):
    """Order of the points of `p` (B, N, 3) by (batch, cell of `grid`)."""
    B, N = p.shape[0], p.shape[1]
    c = torch.floor((p - grid[:, None, :3]) * grid[:, None, 3:]).clamp_(0, G - 1).to(torch.int64)
    key = ((c[..., 0] * G + c[..., 1]) * G + c[..., 2]) + torch.arange(B, device=p.device)[:, None] * (G ** 3)
    skey, perm = torch.sort(key.reshape(-1))
    within = (perm - torch.div(perm, N, rounding_mode="floor") * N).to(torch.int32)
    if not want_start:
        return within
    start = torch.searchsorted(skey, torch.arange(B * G ** 3 + 1, device=p.device)).to(torch.int32)
    return p.reshape(-1, 3)[perm].contiguous(), within, start


def ball_query(points: torch.Tensor, queries: torch.Tensor, radius: float, max_neighbors: int, return_dists: bool = False,
               method: str | None = None):
    """For every query the up to `max_neighbors` nearest points within `radius`, nearest first.

    points (B, Np, 3), queries (B, Nq, 3) -> indices (B, Nq, K) int64 (0 in unused slots), neighbor coordinates
    (B, Nq, K, 3) float32 (zeros in unused slots), counts (B, Nq) int32 [, distances (B, Nq, K)].  Not differentiable:
    callers that need gradients w.r.t. `points` gather them again by the indices.  `method`: "pairs" looks at every
    pair, "cells" bins the points into a uniform grid first (the default from 2048 points on); same results."""
    if not (points.is_cuda and queries.is_cuda):
        raise RuntimeError("physicsnemo_amd kernels need CUDA (ROCm) tensors")
    if points.ndim != 3 or queries.ndim != 3 or points.shape[-1] != 3 or queries.shape[-1] != 3:
        raise ValueError("ball_query needs (B, N, 3) points and queries")
    if points.shape[0] != queries.shape[0]:
        raise ValueError(f"Batch dimensions must match: points has {points.shape[0]}, queries has {queries.shape[0]}")
    pts, qs = points.detach().float().contiguous(), queries.detach().float().contiguous()
    B, Np, Nq, K = pts.shape[0], pts.shape[1], qs.shape[1], int(max_neighbors)
    idx = torch.empty(B, Nq, K, dtype=torch.int64, device=pts.device)
    out = torch.empty(B, Nq, K, 3, dtype=torch.float32, device=pts.device)
    counts = torch.empty(B, Nq, dtype=torch.int32, device=pts.device)
    dists = torch.empty(B, Nq, K, dtype=torch.float32, device=pts.device) if return_dists else None
    method = method or ("cells" if Np >= 2048 else "pairs")
    if method == "cells":
        G = int(min(128, max(2, round((Np / 2.0) ** (1.0 / 3.0)))))  # about two points per cell of a filled box
        while B * G ** 3 >= 2 ** 31:
            G //= 2
        grid, spts, sidx, start = _cell_list(pts, radius, G)
        order = _bin(qs, grid, G, want_start=False) if Nq >= 256 else None
        _lib.check(_lib.load().pa_ball_query_cells(B, Np, Nq, K, float(radius), G, grid.data_ptr(), spts.data_ptr(),
                                                   sidx.data_ptr(), start.data_ptr(), qs.data_ptr(), _lib.ptr(order),
                                                   idx.data_ptr(), out.data_ptr(), _lib.ptr(dists), counts.data_ptr(),
                                                   _lib.current_stream_ptr(pts.device)), "pa_ball_query_cells")
    elif method == "pairs":
        _lib.check(_lib.load().pa_ball_query(B, Np, Nq, K, float(radius), pts.data_ptr(), qs.data_ptr(), idx.data_ptr(),
                                             out.data_ptr(), _lib.ptr(dists), counts.data_ptr(),
                                             _lib.current_stream_ptr(pts.device)), "pa_ball_query")
    else:
        raise ValueError(f"unknown ball_query method {method!r}")
    return (idx, out, counts, dists) if return_dists else (idx, out, counts)
