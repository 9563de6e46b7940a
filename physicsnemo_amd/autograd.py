"""Training path of the PhysicsAttention layer: a torch.autograd.Function whose forward runs the stage-level HIP
kernels and keeps their intermediates, and whose backward runs the backward kernels of libphysattn.so.

The reference has no backward code of its own (autograd differentiates physics_attention.py:501-558 op by op);
this is the same gradient, assembled from
  * hand-written kernels for everything specific to the layer (slice softmax, slice sums, slice attention,
    deslice and their adjoints, the input-gradient GEMMs / transposed convolutions), and
  * the weight gradients ``d out^T . in`` (products over the point axis; for the structured layers against the
    neighbours at every tap) on the library's own MFMA kernels for the shapes they serve, and on the GEMM library
    behind ``torch.matmul`` otherwise (odd widths).
"""
from __future__ import annotations

import functools
import itertools

import torch

from . import functional as PF


def _rows(t: torch.Tensor) -> torch.Tensor:
    return t.reshape(-1, t.shape[-1])


def _aligned(t: torch.Tensor) -> torch.Tensor:
    """`t` itself, or a copy when it is a view that starts off a 16-byte boundary (a batch element of odd size)."""
    t = t.contiguous()
    return t if t.data_ptr() % 16 == 0 else t.clone()


def _wgrad(d_out: torch.Tensor, inp: torch.Tensor):
    """(d W, d b) = (d out^T . in, column sums of d out) over all rows: one pass of the library's MFMA kernel where it
    serves the shape, else the GEMM library and a reduction."""
    d_out, inp = d_out.contiguous(), inp.contiguous()
    served = PF.try_cols_gemm(d_out, inp)
    if served is not None:
        return served
    ca, cb = d_out.shape[-1], inp.shape[-1]
    rows = d_out.numel() // ca
    fold = 32 // ca if ca < 32 and 32 % ca == 0 else 0
    if fold and rows % fold == 0 and d_out.is_contiguous() and inp.is_contiguous():
        # narrow d out (slice_num 16): `fold` consecutive rows side by side make 32 columns; the wanted product is the
        # sum of the diagonal blocks of the folded one
        a2, b2 = d_out.reshape(rows // fold, 32), inp.reshape(rows // fold, cb * fold)
        folded = PF.try_cols_gemm(a2, b2)
        if folded is not None:
            p2, s2 = folded
            dw = sum(p2[k * ca:(k + 1) * ca, k * cb:(k + 1) * cb] for k in range(fold))
            return dw, s2.reshape(fold, ca).sum(0)
    return _rows(d_out).t() @ _rows(inp), _rows(d_out).sum(0, dtype=torch.float32)


def _conv_weight_grad(d_out: torch.Tensor, x: torch.Tensor, dims):
    """(d W, d b) of a grid convolution: d W[o, c, taps...] = sum over grid points of d_out[p, o] * x[p + tap - k//2, c]
    (zero outside the grid), d b[o] = sum d_out[p, o].

    d_out (B, N, O), x (B, N, C) channels-last over the grid of `dims`.  One pass of the library's kernel where it serves
    the widths; otherwise the GEMM library on the unfolded input (2-D) or tap by tap."""
    served = PF.try_cols_gemm(d_out, x, dims)
    if served is not None:
        return served
    k = dims.conv_k
    grid = (dims.grid_h, dims.grid_w) + ((dims.grid_d,) if dims.grid_d > 0 else ())
    d_b = _rows(d_out).sum(0, dtype=torch.float32)
    B, O, C, nd, pad = x.shape[0], d_out.shape[-1], x.shape[-1], len(grid), k // 2
    if nd == 2:
        # one product against the unfolded (im2col) input: its columns are ordered (c, u, v) like the weight
        cols = torch.nn.functional.unfold(x.reshape(B, *grid, C).permute(0, 3, 1, 2), k, padding=pad)  # (B, C k k, N)
        return (_rows(d_out).t() @ cols.transpose(1, 2).reshape(-1, C * k * k)).reshape(O, C, k, k), d_b
    dg, xg = d_out.reshape(B, *grid, O), x.reshape(B, *grid, C)
    dW = torch.zeros((O, C) + (k,) * nd, dtype=d_out.dtype, device=x.device)
    for tap in itertools.product(range(k), repeat=nd):
        lo = [max(0, pad - u) for u in tap]
        hi = [min(g, g + pad - u) for g, u in zip(grid, tap)]
        if any(a >= b for a, b in zip(lo, hi)):
            continue
        out_sl = (slice(None),) + tuple(slice(a, b) for a, b in zip(lo, hi))
        in_sl = (slice(None),) + tuple(slice(a + u - pad, b + u - pad) for a, b, u in zip(lo, hi, tap))
        dW[(slice(None), slice(None)) + tap] = dg[out_sl].reshape(-1, O).t() @ xg[in_sl].reshape(-1, C)
    return dW, d_b


def _torch_conv_layout(w_flat: torch.Tensor, O: int, C: int, taps: tuple, dims) -> torch.Tensor:
    """The kernel-form convolution weight (flat; tap-major when `dims.conv_tap_major`) as torch's (O, C, k, ...)."""
    if dims.conv_tap_major:
        return w_flat.view(O, *taps, C).movedim(-1, 1)
    return w_flat.view(O, C, *taps)


def _slice_weight_grad(d_z: torch.Tensor, x_mid: torch.Tensor, H: int, S: int, D: int):
    """d W_slice[s, d] = sum over points and heads of d z[n, h, s] x_mid[n, h, d] (+ d b_slice).

    As a product over (point, head) rows the operands are only S and D wide, which leaves the row-axis kernel two waves
    per workgroup; taking whole points as rows ((H S) x (H D) result) fills it, and the wanted sum is the sum of the H
    diagonal blocks -- 8 x the arithmetic on matrix cores that have the slack, 30 % less time."""
    a, b = d_z.reshape(-1, H * S), x_mid.reshape(-1, H * D)
    if H > 1 and H * S <= 512 and PF.cols_gemm_supported(a, b):  # wider: the extra passes over x_mid cost more
        p, sums = PF.cols_gemm(a, b, col_sums=True)
        dw = p.view(H, S, H, D).diagonal(dim1=0, dim2=2).sum(-1)
        return dw, sums.reshape(H, S).sum(0)
    return _wgrad(d_z.reshape(-1, S), x_mid.reshape(-1, D))


def _finish_backward(ctx, x, dy, out_x, d_wqkv, d_proj, d_z, d_temp, x_mid, temperature, param_offset=3, slice_grads=None,
                     out_grads=None):
    """Everything after the layer-specific kernels: d x (input-gradient GEMM / transposed convolution) and the weight
    and bias gradients, which are plain GEMMs / column sums over the point axis.  Returns (d x, None, None, the ten
    parameter gradients); `param_offset`: position of the first parameter among the Function's inputs.  `slice_grads`,
    `out_grads`: (d weight, d bias) of in_project_slice (with d temperature masked) and of out_linear where the kernels
    before this left them."""
    dims, kp = ctx.dims, ctx.kparams
    B, N, C, H, D, S = dims.B, dims.N, dims.C, dims.H, dims.D, dims.S
    HD = H * D
    linear = PF.LayerDims(B, N, C, H, D, S)
    if out_grads is not None:
        d_wo, d_bo = out_grads
    else:
        d_wo, d_bo = _wgrad(dy, out_x) if out_x is not None else (None, None)  # None: no out_linear (context projector)
    if slice_grads is not None:
        d_ws, d_bs = slice_grads
    else:
        d_ws, d_bs = _slice_weight_grad(d_z, x_mid, H, S, D)
        t = temperature.reshape(-1)
        d_temp = d_temp * ((t >= 0.5) & (t <= 5.0)).to(d_temp.dtype)

    k = dims.conv_k
    wx, wf = kp["in_project_x_weight"], kp["in_project_fx_weight"]
    if k == 0:
        w_cat = torch.cat([wx.view(HD, C).t(), wf.view(HD, C).t()], dim=1).contiguous()  # (C, 2HD)
        dx = PF.rows_gemm(d_proj, w_cat, None, linear, 2 * HD, C) if ctx.needs_input_grad[0] else None
        d_w_in, d_b_in = _wgrad(d_proj, x)  # (2HD, C), (2HD)
    else:
        grid = (dims.grid_h, dims.grid_w) + ((dims.grid_d,) if dims.grid_d > 0 else ())
        taps = (k,) * len(grid)
        w_both = torch.cat([_torch_conv_layout(wx, HD, C, taps, dims), _torch_conv_layout(wf, HD, C, taps, dims)],
                           dim=0)  # (2HD, C, k, ...)
        # transposed convolution = the same gather with flipped taps and swapped channel roles
        w_t = w_both.flip(dims=tuple(range(2, 2 + len(grid)))).transpose(0, 1)  # (C, 2HD, k, ...)
        w_t = (w_t.movedim(1, -1) if dims.conv_tap_major else w_t).contiguous()
        dx = PF.rows_gemm(d_proj, w_t, None, dims, 2 * HD, C) if ctx.needs_input_grad[0] else None
        d_w_in, d_b_in = _conv_weight_grad(d_proj, x, dims)

    grads = (d_w_in[:HD], d_b_in[:HD], d_w_in[HD:], d_b_in[HD:], d_ws, d_bs, d_temp, d_wqkv, d_wo, d_bo)
    grads = tuple(gr.reshape(p.shape).to(p.dtype) if gr is not None and ctx.needs_input_grad[param_offset + i] else None
                  for i, (gr, p) in enumerate(zip(grads, ctx.param_like)))
    return (dx, None, None) + grads


class PhysicsAttentionFunction(torch.autograd.Function):
    """y = PhysicsAttention(x); differentiable w.r.t. x and the ten parameters.  General kernels (any shape, fp32 or
    bf16 storage): the forward keeps x_mid, fx_mid, the slice weights, the slice tokens and out_x."""

    @staticmethod
    def forward(ctx, x, dims, kparams, wx, bx, wf, bf, ws, bs, temperature, wqkv, wo, bo):
        x_mid, fx_mid = PF.project_inputs(x, kparams, dims)
        w = PF.slice_softmax(x_mid, kparams, dims)
        tok, norm = PF.slice_reduce(w, fx_mid, dims)
        tok_out = PF.slice_attention(tok, kparams, dims)
        y, out_x = PF.deslice_project(w, tok_out, kparams, dims, return_out_x=True)
        ctx.save_for_backward(x, x_mid, fx_mid, w, tok, norm, tok_out, out_x, temperature)
        ctx.dims, ctx.kparams = dims, kparams
        ctx.param_like = (wx, bx, wf, bf, ws, bs, temperature, wqkv, wo, bo)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, x_mid, fx_mid, w, tok, norm, tok_out, out_x, temperature = ctx.saved_tensors
        dims, kp = ctx.dims, ctx.kparams
        C, HD, D = dims.C, dims.H * dims.D, dims.D
        dy = dy.to(x.dtype).contiguous()
        linear = PF.LayerDims(dims.B, dims.N, C, dims.H, D, dims.S)
        # out_linear: g = d out_x
        g = PF.rows_gemm(dy, kp["out_linear_weight"].view(C, HD).t().contiguous(), None, linear, C, HD)
        # adjoint of the deslice w.r.t. the attended tokens, then the slice attention and the normalisation
        d_tok_out = PF.slice_weighted_sum(w, g, dims)[..., :D].contiguous()
        d_num, d_norm, d_wqkv = PF.slice_attention_backward(tok, norm, d_tok_out, kp, dims)
        # per point: slice softmax, aggregation and deslice adjoints
        d_proj, d_z, d_temp = PF.slice_softmax_backward(x_mid, fx_mid, w, g, tok_out, d_num, d_norm, kp, dims)
        return _finish_backward(ctx, x, dy, out_x, d_wqkv, d_proj, d_z, d_temp, x_mid, temperature)


_LAYER_PARAMS = ("in_project_x_weight", "in_project_x_bias", "in_project_fx_weight", "in_project_fx_bias",
                 "in_project_slice_weight", "in_project_slice_bias", "temperature", "qkv_project_weight",
                 "out_linear_weight", "out_linear_bias")
_PLUS_PARAMS = ("in_project_x_weight", "in_project_x_bias", "in_project_slice_weight", "in_project_slice_bias", "temperature",
                "proj_temperature_0_weight", "proj_temperature_0_bias", "proj_temperature_2_weight",
                "proj_temperature_2_bias", "qkv_project_weight", "out_linear_weight", "out_linear_bias")
_LARGE = ("in_project_x_weight", "in_project_fx_weight", "out_linear_weight")


def _train_params(names, params, device, dtype=torch.bfloat16):
    """The parameters as `layer_train_forward` takes them for an input of `dtype`: on the input's device, each on a 16-byte
    boundary (a view into one flat vector of all parameters need not start on one)."""
    as_they_are = dtype == torch.bfloat16 and all(p.dtype == torch.bfloat16 for n, p in zip(names, params) if n in _LARGE)
    large = torch.bfloat16 if as_they_are else torch.float32
    out = {}
    for n, p in zip(names, params):
        wanted = large if n in _LARGE else torch.float32
        if p.dtype != wanted or p.device != device:
            p = p.detach().to(device=device, dtype=wanted)
        out[n] = _aligned(p)
    return out


def _layer_train_forward(ctx, x, uniform, dims, names, params):
    """Forward of a bf16 layer with 32-wide heads in one library call; ctx keeps what the backward call reads."""
    x, uniform = _aligned(x), None if uniform is None else _aligned(uniform)
    y, saved = PF.layer_train_forward(x, uniform, _train_params(names, params, x.device, x.dtype), dims)
    ctx.save_for_backward(x, uniform, saved)
    ctx.dims, ctx.names, ctx.like = dims, names, _shapes_and_types(params)
    return y


# where a parameter's gradient lies among those of the library call
_GRADIENT_ORDER = {names: ([names.index(n) for n in order], [order.index(n) for n in names]) for names, order in
                   ((_LAYER_PARAMS, PF.TRAIN_GRADIENTS), (_PLUS_PARAMS, PF.TRAIN_GRADIENTS_PLUS))}


def _shapes_and_types(params):
    """What the backward pass is to know of the parameters, as they are now: by then they may have been freed, moved or cast."""
    return tuple(p.shape for p in params), tuple(p.dtype for p in params)


@functools.lru_cache(maxsize=64)
def _of_shapes(shapes):  # tensors without memory, for a call that takes shapes as tensors
    return [torch.empty(s, device="meta") for s in shapes]


def _layer_train_backward(ctx, x, uniform, dy, saved, need):
    """(dx, the parameters' gradients); need: which of them are wanted."""
    dx, grads = PF.layer_train_gradients(x, uniform, dy, saved, ctx.dims, ctx.needs_input_grad[0])
    to_buffer, from_buffer = _GRADIENT_ORDER[ctx.names]
    shapes, dtypes = ctx.like
    views = torch._utils._unflatten_dense_tensors(grads, _of_shapes(tuple(shapes[k] for k in to_buffer)))
    out = []
    for dtype, k, wanted in zip(dtypes, from_buffer, need):
        g = views[k] if wanted else None
        out.append(g if g is None or dtype == torch.float32 else g.to(dtype))
    return dx, tuple(out)


class PhysicsAttentionMfmaFunction(torch.autograd.Function):
    """The same gradient in one library call forward and one backward (bf16 MFMA kernels for 32-wide heads, the general kernels
    for float32; irregular and structured variants); the parameters go to the library as they are (`kparams` is not read)."""

    @staticmethod
    def forward(ctx, x, dims, kparams, *params):
        return _layer_train_forward(ctx, x, None, dims, _LAYER_PARAMS, params)

    @staticmethod
    def backward(ctx, dy):
        x, uniform, saved = ctx.saved_tensors
        dx, grads = _layer_train_backward(ctx, x, uniform, _aligned(dy.to(x.dtype)), saved, ctx.needs_input_grad[3:])
        return (dx, None, None) + grads


def _keep_parameters(ctx, *params):
    """For a backward pass that is differentiated again: the parameters themselves, where the saved tensors are copies in the
    kernels' type.  They are not saved tensors, so that changing one between the passes stays allowed without that."""
    ctx.kept = [(p, None if p.is_inference() else p._version) for p in params]


def _kept_parameters(ctx):
    if any(version is not None and p._version != version for p, version in ctx.kept):
        raise RuntimeError("a parameter was modified in place between the forward and a backward pass with create_graph=True")
    return [p for p, _ in ctx.kept]


def _layernorm_backward(ctx, x, dy, w32, eps, add=None):
    """(dx, d weight, d bias) of LayerNorm, dx with `add`: the library's kernel, or the same formulas as tensor ops on the kept
    weight where the result is differentiated again."""
    if not torch.is_grad_enabled():
        return PF.layernorm_backward(x, dy, w32, eps, add)
    return _layernorm_grad_ops(x, dy, _kept_parameters(ctx)[-1], eps, add)


def _layernorm_grad_ops(x, dy, weight, eps, add=None):
    """(dx + add, d weight, d bias) of LayerNorm as tensor operations that can be differentiated again."""
    xf, df = x.float(), dy.float()
    centred = xf - xf.mean(-1, keepdim=True)
    rstd = torch.rsqrt(centred.square().mean(-1, keepdim=True) + eps)
    xh, g = centred * rstd, df * weight.float()
    dx = rstd * (g - g.mean(-1, keepdim=True) - xh * (g * xh).mean(-1, keepdim=True))
    return (dx if add is None else dx + add.float()).to(x.dtype), _rows(df * xh).sum(0), _rows(df).sum(0)


def _through_norm(ctx, y, w32, d_y, d_normed):
    """(gradient of y, d weight, d bias) for the outputs y and LayerNorm(y)."""
    if d_normed is None:
        return (None if d_y is None else _aligned(d_y.to(y.dtype))), None, None
    add = None if d_y is None else _aligned(d_y.to(y.dtype))
    d, dg, db = _layernorm_backward(ctx, y, _aligned(d_normed.to(y.dtype)), w32, ctx.eps, add)
    return d, dg.to(ctx.ln_dtypes[0]), db.to(ctx.ln_dtypes[1])


class LayerResidualNormFunction(torch.autograd.Function):
    """(y, LayerNorm(y)) for y = layer(x) + residual: `PhysicsAttentionMfmaFunction` with the block's residual and
    following LayerNorm in the forward's last kernel, and the residual's gradient in the LayerNorm's backward kernel."""

    @staticmethod
    def forward(ctx, x, residual, dims, ln_w, ln_b, eps, *params):
        ctx.set_materialize_grads(False)
        w32 = _aligned(ln_w.detach().float())
        kernel_params = _train_params(_LAYER_PARAMS, params, x.device, x.dtype)
        y, saved, normed = PF.layer_train_forward(x, None, kernel_params, dims, residual, w32, _aligned(ln_b.detach().float()), eps)
        ctx.save_for_backward(x, saved, y, w32)
        ctx.dims, ctx.names, ctx.like = dims, _LAYER_PARAMS, _shapes_and_types(params)
        ctx.eps, ctx.ln_dtypes = eps, (ln_w.dtype, ln_b.dtype)
        _keep_parameters(ctx, ln_w)
        return y, normed

    @staticmethod
    def backward(ctx, d_y, d_normed):
        x, saved, y, w32 = ctx.saved_tensors
        need = ctx.needs_input_grad
        d, dg, db = _through_norm(ctx, y, w32, d_y, d_normed)
        if d is None:
            return (None,) * (6 + len(_LAYER_PARAMS))
        dx, grads = _layer_train_backward(ctx, x, None, d, saved, need[6:])
        return (dx, d if need[1] else None, None, dg, db, None) + grads


class LayerResidualFunction(torch.autograd.Function):
    """(y, LayerNorm(y)) as `LayerResidualNormFunction`, the second without a gradient of its own: for a consumer that takes
    both and differentiates the LayerNorm itself (`NormMlpResidualFunction`)."""

    @staticmethod
    def forward(ctx, x, residual, dims, ln_w, ln_b, eps, *params):
        ctx.set_materialize_grads(False)
        kernel_params = _train_params(_LAYER_PARAMS, params, x.device, x.dtype)
        y, saved, normed = PF.layer_train_forward(x, None, kernel_params, dims, residual,
                                                  _aligned(ln_w.detach().float()), _aligned(ln_b.detach().float()), eps)
        ctx.save_for_backward(x, saved)
        ctx.dims, ctx.names, ctx.like = dims, _LAYER_PARAMS, _shapes_and_types(params)
        ctx.mark_non_differentiable(normed)
        return y, normed

    @staticmethod
    def backward(ctx, d_y, _):
        x, saved = ctx.saved_tensors
        need = ctx.needs_input_grad
        if d_y is None:
            return (None,) * (6 + len(_LAYER_PARAMS))
        d = _aligned(d_y.to(x.dtype))
        dx, grads = _layer_train_backward(ctx, x, None, d, saved, need[6:])
        return (dx, d if need[1] else None, None, None, None, None) + grads


class PhysicsAttentionPlusMfmaFunction(torch.autograd.Function):
    """`PhysicsAttentionPlusFunction` on the bf16 MFMA kernels (32-wide heads)."""

    @staticmethod
    def forward(ctx, x, uniform, dims, *params):
        return _layer_train_forward(ctx, x, uniform, dims, _PLUS_PARAMS, params)

    @staticmethod
    def backward(ctx, dy):
        x, uniform, saved = ctx.saved_tensors
        dx, grads = _layer_train_backward(ctx, x, uniform, _aligned(dy.to(x.dtype)), saved, ctx.needs_input_grad[3:])
        return (dx, None, None) + grads


def _plus_backward_tail(ctx, x, uniform, x_mid, w, tok_out, out_x, dy, g, d_num, d_norm, d_wqkv, first_param):
    """Everything of the Transolver++ backward after the slice-token stage: the per-point kernel, d x and the parameter
    gradients (d_wqkv is passed through; None when the caller's token-stage graph provides it).  Returns (d x, the
    twelve parameter gradients in the order of `ctx.param_like`)."""
    dims, kp = ctx.dims, ctx.kparams
    B, N, C, H, D, S = dims.B, dims.N, dims.C, dims.H, dims.D, dims.S
    HD = H * D
    linear = PF.LayerDims(B, N, C, H, D, S)
    d_xm, d_z, d_a1, d_a2, d_temp = PF.slice_softmax_plus_backward(x_mid, uniform, w, g, tok_out, d_num, d_norm, kp, dims)
    d_wo, d_bo = _wgrad(dy, out_x)
    xm_rows = x_mid.reshape(-1, D)
    d_ws, d_bs = _wgrad(d_z.reshape(-1, S), xm_rows)
    # proj_temperature = Linear(D, S) -> GELU -> Linear(S, 1) -> GELU: the kernel returns the gradients of the two
    # Linear outputs; the second weight gradient needs the hidden activation again
    d_w1, d_b1 = _wgrad(d_a1.reshape(-1, S), xm_rows)
    hidden = torch.nn.functional.gelu(torch.addmm(kp["proj_temperature_0_bias"], xm_rows.float(),
                                                  kp["proj_temperature_0_weight"].view(S, D).t()))
    d_w2 = (d_a2.reshape(-1, 1) * hidden).sum(0, keepdim=True)  # (1, rows) x (rows, S): a reduction, not a GEMM shape
    d_b2 = d_a2.sum().reshape(1)

    k = dims.conv_k
    wx = kp["in_project_x_weight"]
    if k == 0:
        dx = PF.rows_gemm(d_xm, wx.view(HD, C).t().contiguous(), None, linear, HD, C) if ctx.needs_input_grad[0] else None
        d_wx, d_bx = _wgrad(d_xm, x)
    else:
        grid = (dims.grid_h, dims.grid_w) + ((dims.grid_d,) if dims.grid_d > 0 else ())
        w_t = _torch_conv_layout(wx, HD, C, (k,) * len(grid), dims).flip(dims=tuple(range(2, 2 + len(grid)))).transpose(0, 1)
        w_t = (w_t.movedim(1, -1) if dims.conv_tap_major else w_t).contiguous()
        dx = PF.rows_gemm(d_xm, w_t, None, dims, HD, C) if ctx.needs_input_grad[0] else None
        d_wx, d_bx = _conv_weight_grad(d_xm, x, dims)

    grads = (d_wx, d_bx, d_ws, d_bs, d_temp, d_w1, d_b1, d_w2, d_b2, d_wqkv, d_wo, d_bo)
    grads = tuple(gr.reshape(p.shape).to(p.dtype) if gr is not None and ctx.needs_input_grad[first_param + i] else None
                  for i, (gr, p) in enumerate(zip(grads, ctx.param_like)))
    return dx, grads


class PhysicsAttentionPlusFunction(torch.autograd.Function):
    """Transolver++ (plus=True) layer, differentiable w.r.t. x and its twelve parameters; general kernels.  ``uniform``
    (B, N, H, S) holds the samples behind the Gumbel noise and gets no gradient (the reference draws them with
    ``torch.rand_like``, gumbel_softmax.py:50)."""

    @staticmethod
    def forward(ctx, x, uniform, dims, kparams, wx, bx, ws, bs, temperature, pt_w1, pt_b1, pt_w2, pt_b2, wqkv, wo, bo):
        x_mid, _ = PF.project_inputs(x, kparams, dims)
        w = PF.slice_softmax_plus(x_mid, uniform, kparams, dims)
        tok, norm = PF.slice_reduce(w, x_mid, dims)
        tok_out = PF.slice_attention(tok, kparams, dims)
        y, out_x = PF.deslice_project(w, tok_out, kparams, dims, return_out_x=True)
        ctx.save_for_backward(x, uniform, x_mid, w, tok, norm, tok_out, out_x)
        ctx.dims, ctx.kparams = dims, kparams
        ctx.param_like = (wx, bx, ws, bs, temperature, pt_w1, pt_b1, pt_w2, pt_b2, wqkv, wo, bo)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, uniform, x_mid, w, tok, norm, tok_out, out_x = ctx.saved_tensors
        dims, kp = ctx.dims, ctx.kparams
        C, HD, D = dims.C, dims.H * dims.D, dims.D
        dy = dy.to(x.dtype).contiguous()
        linear = PF.LayerDims(dims.B, dims.N, C, dims.H, D, dims.S)
        g = PF.rows_gemm(dy, kp["out_linear_weight"].view(C, HD).t().contiguous(), None, linear, C, HD)
        d_tok_out = PF.slice_weighted_sum(w, g, dims)[..., :D].contiguous()
        d_num, d_norm, d_wqkv = PF.slice_attention_backward(tok, norm, d_tok_out, kp, dims)
        dx, grads = _plus_backward_tail(ctx, x, uniform, x_mid, w, tok_out, out_x, dy, g, d_num, d_norm, d_wqkv, 4)
        return (dx, None, None, None) + grads


class GALEPlusFunction(torch.autograd.Function):
    """Transolver++ form of the GALE layer with a context (gale.py:148-239 with plus=True): the per-point stages of
    `PhysicsAttentionPlusFunction`, the slice-token stage (self-attention, cross-attention, blend) as a PyTorch graph
    like in `GALEFunction`.  Differentiable w.r.t. x, the context, the twelve layer parameters and the stage's."""

    @staticmethod
    def forward(ctx, x, uniform, context, dims, kparams, token_stage, n_stage, *params):
        layer_params, stage_params = params[:len(params) - n_stage], params[len(params) - n_stage:]
        x_mid, _ = PF.project_inputs(x, kparams, dims)
        w = PF.slice_softmax_plus(x_mid, uniform, kparams, dims)
        tok, norm = PF.slice_reduce(w, x_mid, dims)
        with torch.enable_grad():
            tok_leaf = tok.detach().requires_grad_(True)
            ctx_leaf = context.detach().requires_grad_(ctx.needs_input_grad[2])
            out_graph = token_stage(tok_leaf, ctx_leaf)
        tok_out = out_graph.detach().float().contiguous()
        y, out_x = PF.deslice_project(w, tok_out, kparams, dims, return_out_x=True)
        ctx.save_for_backward(x, uniform, x_mid, w, tok, norm, tok_out, out_x)
        ctx.dims, ctx.kparams = dims, kparams
        ctx.param_like = layer_params
        ctx.graph = (out_graph, tok_leaf, ctx_leaf, stage_params)
        return y

    @staticmethod
    def backward(ctx, dy):
        x, uniform, x_mid, w, tok, norm, tok_out, out_x = ctx.saved_tensors
        dims, kp = ctx.dims, ctx.kparams
        C, HD, D = dims.C, dims.H * dims.D, dims.D
        dy = dy.to(x.dtype).contiguous()
        linear = PF.LayerDims(dims.B, dims.N, C, dims.H, D, dims.S)
        g = PF.rows_gemm(dy, kp["out_linear_weight"].view(C, HD).t().contiguous(), None, linear, C, HD)
        d_tok_out = PF.slice_weighted_sum(w, g, dims)[..., :D].contiguous()
        out_graph, tok_leaf, ctx_leaf, stage_params = ctx.graph
        wanted = [tok_leaf] + ([ctx_leaf] if ctx_leaf.requires_grad else []) + \
                 [p for p in stage_params if p.requires_grad]
        got = list(torch.autograd.grad(out_graph, wanted, d_tok_out.to(out_graph.dtype), allow_unused=True))
        d_tok = got.pop(0).float()
        d_context = got.pop(0) if ctx_leaf.requires_grad else None
        d_stage = [got.pop(0) if p.requires_grad else None for p in stage_params]
        d_num = (d_tok / norm[..., None]).contiguous()
        d_norm = (-(d_tok * tok).sum(-1) / norm).contiguous()
        # qkv_project.weight takes part in the token stage only: its gradient comes with `d_stage`
        dx, grads = _plus_backward_tail(ctx, x, uniform, x_mid, w, tok_out, out_x, dy, g, d_num, d_norm, None, 7)
        return (dx, None, d_context, None, None, None, None) + grads + tuple(d_stage)


class GALEFunction(torch.autograd.Function):
    """GALE layer with a context (gale.py:148-239), differentiable w.r.t. x, the context, the ten PhysicsAttention
    parameters and the cross-attention / blend parameters.

    The per-point stages are the layer's kernels, forward and backward, as in the two Functions above.  The slice-token
    stage in between (self-attention, cross-attention to the context, blend: S x D work per (batch, head), independent
    of the number of points) is evaluated by `token_stage(tok, context)` with PyTorch ops under autograd in the
    forward; the backward asks that small graph for d tok, d context and the gradients of `stage_params`."""

    @staticmethod
    def forward(ctx, x, context, dims, kparams, token_stage, n_stage, *params):
        layer_params, stage_params = params[:len(params) - n_stage], params[len(params) - n_stage:]
        mfma = PF.mfma_backward_supported(x.dtype, dims)
        if mfma:
            st = PF.MfmaStages(kparams, dims, x.device)
            st.pack_params()
            if st.fused_groups > 0:
                st.project_softmax_reduce(x)
            else:
                st.project_softmax(x)
                st.slice_reduce()
            st.combine_attention()  # for the normalised slice tokens; its self-attention result is replaced below
            tok, norm = st.tok, st.norm
        else:
            x_mid, fx_mid = PF.project_inputs(x, kparams, dims)
            w = PF.slice_softmax(x_mid, kparams, dims)
            tok, norm = PF.slice_reduce(w, fx_mid, dims)
        with torch.enable_grad():
            tok_leaf = tok.detach().requires_grad_(True)
            ctx_leaf = context.detach().requires_grad_(ctx.needs_input_grad[1])
            out_graph = token_stage(tok_leaf, ctx_leaf)
        out_tok = out_graph.detach().float().contiguous()
        if mfma:
            st.set_out_tokens(out_tok)
            y = torch.empty_like(x)
            st.deslice_project(y)
            ctx.save_for_backward(x, layer_params[6])
            ctx.stages = st
        else:
            y, out_x = PF.deslice_project(w, out_tok, kparams, dims, return_out_x=True)
            ctx.save_for_backward(x, layer_params[6], x_mid, fx_mid, w, out_x)
        ctx.mfma, ctx.dims, ctx.kparams = mfma, dims, kparams
        ctx.tok, ctx.norm, ctx.out_tok = tok, norm, out_tok
        ctx.graph = (out_graph, tok_leaf, ctx_leaf, stage_params)
        ctx.param_like = layer_params
        return y

    @staticmethod
    def backward(ctx, dy):
        dims, kp = ctx.dims, ctx.kparams
        C, HD, D = dims.C, dims.H * dims.D, dims.D
        x, temperature = ctx.saved_tensors[:2]
        dy = dy.to(x.dtype).contiguous()
        linear = PF.LayerDims(dims.B, dims.N, C, dims.H, D, dims.S)
        w_out_t = kp["out_linear_weight"].view(C, HD).t().contiguous()
        g = PF.rows_gemm(dy, w_out_t, None, linear, C, HD)
        if ctx.mfma:
            st = ctx.stages
            x_mid, fx_mid = PF.project_inputs(x, kp, dims)
            d_out_tok, d_wo, d_bo = PF.output_backward(st.w_pack, dy, ctx.out_tok, kp["out_linear_weight"], dims)
        else:
            x_mid, fx_mid, w, out_x = ctx.saved_tensors[2:]
            d_out_tok = PF.slice_weighted_sum(w, g, dims)[..., :D].contiguous()
        # slice-token stage: PyTorch's graph of the forward
        out_graph, tok_leaf, ctx_leaf, stage_params = ctx.graph
        wanted = [tok_leaf] + ([ctx_leaf] if ctx_leaf.requires_grad else []) + \
                 [p for p in stage_params if p.requires_grad]
        got = list(torch.autograd.grad(out_graph, wanted, d_out_tok.to(out_graph.dtype), allow_unused=True))
        d_tok = got.pop(0).float()
        d_context = got.pop(0) if ctx_leaf.requires_grad else None
        d_stage = [got.pop(0) if p.requires_grad else None for p in stage_params]
        # tok = num / nrm
        d_num = (d_tok / ctx.norm[..., None]).contiguous()
        d_norm = (-(d_tok * ctx.tok).sum(-1) / ctx.norm).contiguous()
        # qkv_project.weight takes part in the token stage only: its gradient comes with `d_stage`
        if ctx.mfma:
            d_proj, d_ws, d_bs, d_temp = PF.point_backward(x_mid, fx_mid, g, ctx.out_tok, d_num, d_norm, kp, dims)
            base = _finish_backward(ctx, x, dy, None, None, d_proj, None, d_temp, x_mid, temperature, 6, (d_ws, d_bs), (d_wo, d_bo))
        else:
            d_proj, d_z, d_temp = PF.slice_softmax_backward(x_mid, fx_mid, w, g, ctx.out_tok, d_num, d_norm, kp, dims)
            base = _finish_backward(ctx, x, dy, out_x, None, d_proj, d_z, d_temp, x_mid, temperature, param_offset=6)
        return (base[0], d_context, None, None, None, None) + base[3:] + tuple(d_stage)


class SliceTokensFunction(torch.autograd.Function):
    """x -> normalised slice tokens (B,H,S,D) float32: the projection, slice-softmax and aggregation stages of the
    layer on their own (a GeoTransolver context projector, context_projector.py:338-378), differentiable w.r.t. x and
    the seven parameters involved.  The backward is the per-point backward kernel with no deslice term (d out_x = 0)."""

    @staticmethod
    def forward(ctx, x, dims, kparams, wx, bx, wf, bf, ws, bs, temperature):
        mfma = PF.mfma_backward_supported(x.dtype, dims)
        if mfma:
            st = PF.MfmaStages(kparams, dims, x.device)
            st.pack_params()
            if st.fused_groups > 0:
                st.project_softmax_reduce(x)
            else:
                st.project_softmax(x)
                st.slice_reduce()
            st.combine_attention()
            tok, norm = st.tok.clone(), st.norm
            ctx.save_for_backward(x, temperature, tok, norm)
        else:
            x_mid, fx_mid = PF.project_inputs(x, kparams, dims)
            w = PF.slice_softmax(x_mid, kparams, dims)
            tok, norm = PF.slice_reduce(w, fx_mid, dims)
            ctx.save_for_backward(x, temperature, tok, norm, x_mid, fx_mid, w)
        ctx.mfma, ctx.dims, ctx.kparams = mfma, dims, kparams
        ctx.param_like = (wx, bx, wf, bf, ws, bs, temperature)
        return tok

    @staticmethod
    def backward(ctx, d_tok):
        dims, kp = ctx.dims, ctx.kparams
        x, temperature, tok, norm = ctx.saved_tensors[:4]
        d_tok = d_tok.float()
        d_num = (d_tok / norm[..., None]).contiguous()
        d_norm = (-(d_tok * tok).sum(-1) / norm).contiguous()
        g = torch.zeros(dims.B, dims.N, dims.H * dims.D, dtype=x.dtype, device=x.device)
        if ctx.mfma:
            x_mid, fx_mid = PF.project_inputs(x, kp, dims)
            d_proj, d_ws, d_bs, d_temp = PF.point_backward(x_mid, fx_mid, g, None, d_num, d_norm, kp, dims)
            base = _finish_backward(ctx, x, None, None, None, d_proj, None, d_temp, x_mid, temperature, 3, (d_ws, d_bs))
        else:
            x_mid, fx_mid, w = ctx.saved_tensors[4:]
            d_proj, d_z, d_temp = PF.slice_softmax_backward(x_mid, fx_mid, w, g, torch.zeros_like(tok), d_num, d_norm,
                                                            kp, dims)
            base = _finish_backward(ctx, x, None, None, None, d_proj, d_z, d_temp, x_mid, temperature)
        return base[:3] + base[3:10]


class FlareFunction(torch.autograd.Function):
    """FLARE layer core (flare_attention.py:38-72, :222-255) given the composed score / value weights: differentiable
    w.r.t. x, the four composed tensors and out_linear.  The composition itself (q_global, self_k / self_v and
    in_project_x folded into two matrices) is a handful of small tensor products done by the caller under autograd, so
    the gradients reach the layer's own parameters through it.  Without out_linear (`wo` None) the result is the
    attention output (B, N, H*D) itself, for callers that blend it with something else first (GALE_FA)."""

    @staticmethod
    def forward(ctx, x, dims, w_a, b_a, w_v, b_v, wo, bo):
        B, N, C, H, D, S = dims.B, dims.N, dims.C, dims.H, dims.D, dims.S
        wa_k, wv_k = w_a.detach().to(x.dtype).contiguous(), w_v.detach().to(x.dtype).contiguous()
        scores = PF.rows_gemm(x, wa_k, b_a.detach().float().contiguous(), dims, C, H * S).view(B, N, H, S)
        values = PF.rows_gemm(x, wv_k, b_v.detach().float().contiguous(), dims, C, H * D)
        col_w, _ = PF.flare_column_weights(scores, dims)
        tok, norm = PF.slice_reduce(col_w, values, dims)
        den = norm - 1e-2  # the aggregation kernel adds the PhysicsAttention epsilon to the divisor; FLARE has none
        z = (tok * (norm / den).unsqueeze(-1)).contiguous()
        row_w = PF.flare_softmax_rows_(scores, dims)
        ctx.dims = dims
        ctx.projected = wo is not None
        if not ctx.projected:
            out_x = PF.deslice(row_w, z, dims)
            ctx.save_for_backward(x, row_w, col_w, values, z, den, wa_k, wv_k)
            ctx.dtypes = tuple(t.dtype for t in (w_a, b_a, w_v, b_v))
            return out_x
        kp = {"out_linear_weight": wo.detach().to(x.dtype).contiguous().reshape(-1),
              "out_linear_bias": bo.detach().float().contiguous()}
        y, out_x = PF.deslice_project(row_w, z, kp, dims, return_out_x=True)
        ctx.save_for_backward(x, row_w, col_w, values, z, den, wa_k, wv_k, out_x, kp["out_linear_weight"])
        ctx.dtypes = tuple(t.dtype for t in (w_a, b_a, w_v, b_v, wo, bo))
        return y

    @staticmethod
    def backward(ctx, dy):
        x, row_w, col_w, values, z, den, wa_k, wv_k = ctx.saved_tensors[:8]
        dims = ctx.dims
        B, N, C, H, D, S = dims.B, dims.N, dims.C, dims.H, dims.D, dims.S
        HD, HS = H * D, H * S
        dy = dy.to(x.dtype).contiguous()
        if ctx.projected:
            out_x, wo_k = ctx.saved_tensors[8:]
            g = PF.rows_gemm(dy, wo_k.view(C, HD).t().contiguous(), None, dims, C, HD)
            d_wo, d_bo = _wgrad(dy, out_x)
        else:
            g, d_wo, d_bo = dy, None, None
        d_z = PF.slice_weighted_sum(row_w, g, dims)[..., :D]
        d_num = (d_z / den.unsqueeze(-1)).contiguous()
        d_den = (-(d_z * z).sum(-1) / den).contiguous()
        d_a, d_v = PF.flare_backward_points(row_w, col_w, values, g, z, d_num, d_den, dims)
        d_a = d_a.view(B, N, HS)
        dx = None
        if ctx.needs_input_grad[0]:
            w_cat = torch.cat([wa_k, wv_k], dim=0).t().contiguous()  # (C, HS + HD)
            dx = PF.rows_gemm(torch.cat([d_a, d_v], dim=-1), w_cat, None, dims, HS + HD, C)
        d_wa, d_ba = _wgrad(d_a, x)
        d_wv, d_bv = _wgrad(d_v, x)
        grads = [gr.float().reshape(shape).to(dt) for gr, shape, dt in zip(
            (d_wa, d_ba, d_wv, d_bv, d_wo, d_bo), ((HS, C), (HS,), (HD, C), (HD,), (C, HD), (C,)), ctx.dtypes)]
        if not ctx.projected:
            grads += [None, None]
        return (dx, None, *grads)


class PointCrossFunction(torch.autograd.Function):
    """Cross-attention of every point to a small set of context tokens, scale 1 (GALE_FA, reference gale.py:735-744):
    out[b,n,h,:] = sum_u softmax_u(x[b,n,:] . w_c[b,(h,u),:] + b_c[b,(h,u)]) v[b,h,u,:].  The caller folds in_project_x,
    cross_q and the context's keys into the per-batch score weight `w_c` (B, H*Sc, C) / `b_c` (B, H*Sc) and projects
    the context's values `v` (B, H, Sc, D), all under autograd.  Scores from the row GEMM, the in-place row softmax and
    the deslice kernel; backward: the row-softmax part of the FLARE per-point kernel (gather weights zero), the
    slice-weighted sum for d v, row / column GEMMs for d x and d w_c."""

    @staticmethod
    def forward(ctx, x, dims, w_c, b_c, v):
        B, N, C, H, Sc = dims.B, dims.N, dims.C, dims.H, dims.S
        one = PF.LayerDims(1, N, C, H, dims.D, Sc)
        wk = w_c.detach().to(x.dtype).contiguous()
        bk = b_c.detach().float().contiguous()
        scores = torch.empty(B, N, H, Sc, dtype=x.dtype, device=x.device)
        for b in range(B):  # the score weight holds the batch element's keys
            scores[b] = PF.rows_gemm(_aligned(x[b:b + 1]), _aligned(wk[b]), _aligned(bk[b]), one, C, H * Sc).view(N, H, Sc)
        p = PF.flare_softmax_rows_(scores, dims)
        v32 = v.detach().float().contiguous()
        ctx.save_for_backward(x, p, v32, wk)
        ctx.dims = dims
        ctx.dtypes = (w_c.dtype, b_c.dtype, v.dtype)
        return PF.deslice(p, v32, dims)

    @staticmethod
    def backward(ctx, g):
        x, p, v32, wk = ctx.saved_tensors
        dims = ctx.dims
        B, N, C, H, D, Sc = dims.B, dims.N, dims.C, dims.H, dims.D, dims.S
        g = g.to(x.dtype).contiguous()
        d_v = PF.slice_weighted_sum(p, g, dims)[..., :D]
        zeros_w = torch.zeros_like(p)
        d_s, _ = PF.flare_backward_points(p, zeros_w, g, g, v32, torch.zeros_like(v32),
                                          torch.zeros(B, H, Sc, dtype=torch.float32, device=x.device), dims)
        d_s = d_s.view(B, N, H * Sc)
        one = PF.LayerDims(1, N, C, H, D, Sc)
        dx = torch.empty_like(x) if ctx.needs_input_grad[0] else None
        d_w, d_b = [], []
        for b in range(B):
            if dx is not None:
                dx[b] = PF.rows_gemm(_aligned(d_s[b:b + 1]), _aligned(wk[b].t()), None, one, H * Sc, C)[0]
            dw_b, db_b = _wgrad(_aligned(d_s[b]), _aligned(x[b]))
            d_w.append(dw_b.float())
            d_b.append(db_b.float())
        return (dx, None, torch.stack(d_w).to(ctx.dtypes[0]), torch.stack(d_b).to(ctx.dtypes[1]),
                d_v.to(ctx.dtypes[2]))


class LinearFunction(torch.autograd.Function):
    """torch.nn.functional.linear for the block MLP in bf16 training: the two row GEMMs (forward, input gradient) go to
    the GEMM library, the weight and bias gradients -- products over the huge row axis, where the library's kernels
    leave most of the machine idle -- to the library's row-axis kernels, which also return them in float32."""

    @staticmethod
    def forward(ctx, x, weight, bias):
        w16 = weight.to(x.dtype)
        ctx.save_for_backward(x, w16)
        _keep_parameters(ctx, weight)
        ctx.param_dtypes = (weight.dtype, bias.dtype if bias is not None else None)
        return torch.nn.functional.linear(x, w16, bias.to(x.dtype) if bias is not None else None)

    @staticmethod
    def backward(ctx, dy):
        x, w16 = ctx.saved_tensors
        dy = dy.contiguous()
        again = torch.is_grad_enabled()  # create_graph: tensor ops on the inputs themselves, to be differentiated again
        dx = (dy @ (_kept_parameters(ctx)[0].to(x.dtype) if again else w16)) if ctx.needs_input_grad[0] else None
        dw = db = None
        if ctx.needs_input_grad[1] or ctx.needs_input_grad[2]:
            if again:
                dw, db = _rows(dy).float().t() @ _rows(x).float(), _rows(dy).sum(0, dtype=torch.float32)
            else:
                dw, db = _wgrad(_rows(dy), _rows(x))
            dw = dw.to(ctx.param_dtypes[0])
            db = db.to(ctx.param_dtypes[1]) if ctx.param_dtypes[1] is not None else None
        return dx, dw, db


def linear(x: torch.Tensor, weight: torch.Tensor, bias: torch.Tensor | None) -> torch.Tensor:
    """Differentiable linear layer; on bf16 / float32 GPU tensors the weight gradient runs on the library's kernels."""
    if x.is_cuda and x.dtype in (torch.bfloat16, torch.float32) and x.numel() > 0:
        return LinearFunction.apply(x.contiguous(), weight, bias)
    return torch.nn.functional.linear(x, weight, bias)


def compute_dtype(x: torch.Tensor) -> torch.dtype | None:
    """The type a Linear of x runs in on the library's training path: bfloat16 under bf16 autocast for the types it casts
    (float64 and whole numbers it leaves alone), x's own float32 or bfloat16 without autocast, None where the modules run as
    they are (also under torch.func transforms and forward-mode differentiation, which the library's functions do not take
    part in)."""
    if not x.is_cuda or torch._C._are_functorch_transforms_active() or torch.autograd.forward_ad._current_level >= 0:
        return None
    if torch.is_autocast_enabled("cuda"):
        cast = x.dtype in (torch.float32, torch.bfloat16, torch.float16)
        return torch.bfloat16 if cast and torch.get_autocast_dtype("cuda") == torch.bfloat16 else None
    return x.dtype if x.dtype in (torch.bfloat16, torch.float32) else None


def unhooked(*modules: torch.nn.Module) -> bool:
    """True where calling the modules is their arithmetic and nothing more.  Hooks observe or change a module's values, and
    `torch.nn.utils`' weight and spectral normalisation and pruning form the weight in one."""
    return not any(m._forward_hooks or m._forward_pre_hooks or m._backward_hooks or m._backward_pre_hooks for m in modules)


def _linears_served(dtype: torch.dtype | None, *lins: torch.nn.Module) -> bool:
    """True where `linear` does what calling the modules does in `dtype`; without autocast a Linear refuses an input whose
    type is not its weight's."""
    return dtype is not None and all(type(m) is torch.nn.Linear and unhooked(m) and
                                     (torch.is_autocast_enabled("cuda") or m.weight.dtype == dtype) for m in lins)


def mlp(x: torch.Tensor, layers: torch.nn.Sequential) -> torch.Tensor:
    """Linear -> activation -> Linear in training, as autocast would run it, on `linear`."""
    dtype = compute_dtype(x)
    if len(layers) != 3 or not unhooked(layers) or not _linears_served(dtype, layers[0], layers[2]):
        return layers(x)
    if not torch.is_autocast_enabled("cuda"):
        return linear(layers[1](linear(x, layers[0].weight, layers[0].bias)), layers[2].weight, layers[2].bias)
    with torch.autocast("cuda", enabled=False):
        h = linear(x.to(dtype), layers[0].weight, layers[0].bias)
        return linear(layers[1](h), layers[2].weight, layers[2].bias)


class MlpResidualFunction(torch.autograd.Function):
    """(y, LayerNorm(y)) for y = residual + Linear(gelu(Linear(x))) of a bf16 block, in one kernel that keeps the hidden
    layer on chip (ln_w None: y alone); the backward forms the hidden layer again from x, so nothing of it is kept between
    the passes (2 x 2 F bytes per row)."""

    @staticmethod
    def forward(ctx, x, residual, w1, b1, w2, b2, ln_w, ln_b, eps):
        ctx.set_materialize_grads(False)
        w1_16, w2_16 = (_aligned(w.detach().to(torch.bfloat16)) for w in (w1, w2))
        b1_32, b2_32 = _aligned(b1.detach().to(torch.float32, copy=True)), _aligned(b2.detach().float())  # b1: read again
        ctx.param_dtypes = tuple(p.dtype for p in (w1, b1, w2, b2))
        _keep_parameters(ctx, w1, b1, w2, *(() if ln_w is None else (ln_w,)))
        packed = PF.mlp_pack(w1_16, w2_16)
        if ln_w is None:
            ctx.save_for_backward(x, w1_16, b1_32, w2_16)
            return PF.mlp_forward_packed(x, packed, b1_32, b2_32, residual=residual, train=True)
        w32 = _aligned(ln_w.detach().float())
        y, normed = PF.mlp_forward_packed(x, packed, b1_32, b2_32, residual=residual, ln_weight=w32,
                                          ln_bias=_aligned(ln_b.detach().float()), ln_eps=eps, train=True)
        ctx.save_for_backward(x, w1_16, b1_32, w2_16, y, w32)
        ctx.eps, ctx.ln_dtypes = eps, (ln_w.dtype, ln_b.dtype)
        return y, normed

    @staticmethod
    def backward(ctx, dy, d_normed=None):
        x, w1, b1, w2, *norm = ctx.saved_tensors
        need = ctx.needs_input_grad
        d_ln = (None, None)
        if norm:
            dy, *d_ln = _through_norm(ctx, norm[0], norm[1], dy, d_normed)
        if dy is None:
            return (None,) * 9
        dy16 = _aligned(dy.to(x.dtype))
        again = torch.is_grad_enabled()
        if again:  # create_graph: the same formulas as tensor ops on the parameters, which can be differentiated again
            w1, b1, w2 = (p.to(x.dtype) for p in _kept_parameters(ctx)[:3])
            h = torch.nn.functional.linear(x, w1, b1)
            act, dh = torch.nn.functional.gelu(h), torch.ops.aten.gelu_backward(dy16 @ w2, h)
        else:
            act, dh = PF.mlp_backward(x, dy16, w1, b1, w2)
        product = _wgrad if not again else lambda d, i: (d.float().t() @ i.float(), d.sum(0, dtype=torch.float32))
        dx = dh @ w1 if need[0] else None
        d_w1, d_b1 = product(_rows(dh), _rows(x)) if need[2] or need[3] else (None, None)
        d_w2, d_b2 = product(_rows(dy16), _rows(act)) if need[4] or need[5] else (None, None)
        grads = (g.to(t) if n else None for g, t, n in zip((d_w1, d_b1, d_w2, d_b2), ctx.param_dtypes, need[2:]))
        return (dx, dy if need[1] else None, *grads, *d_ln, None)


class NormMlpResidualFunction(torch.autograd.Function):
    """(y, next LayerNorm(y)) for y = x + Linear(gelu(Linear(LayerNorm(x)))) of a bf16 block (next_w None: y alone), given
    `normed` = LayerNorm(x) from the kernel that formed x; the backward is one library call from dy, x and normed."""

    @staticmethod
    def forward(ctx, x, normed, ln_w, ln_b, eps, w1, b1, w2, b2, next_w, next_b, next_eps):
        ctx.set_materialize_grads(False)
        w1_16, w2_16 = (_aligned(w.detach().to(torch.bfloat16)) for w in (w1, w2))
        b1_32, b2_32 = _aligned(b1.detach().to(torch.float32, copy=True)), _aligned(b2.detach().float())  # b1: read again
        ln_w32 = _aligned(ln_w.detach().to(torch.float32, copy=True))
        ctx.param_dtypes = tuple(p.dtype for p in (w1, b1, w2, b2, ln_w, ln_b))
        _keep_parameters(ctx, ln_w, ln_b, w1, b1, w2, *(() if next_w is None else (next_w,)))
        ctx.norm_eps = eps
        packed = PF.mlp_pack(w1_16, w2_16)
        if next_w is None:
            ctx.save_for_backward(x, normed, w1_16, b1_32, w2_16, ln_w32)
            return PF.mlp_forward_packed(normed, packed, b1_32, b2_32, residual=x, train=True)
        w32 = _aligned(next_w.detach().float())
        y, nxt = PF.mlp_forward_packed(normed, packed, b1_32, b2_32, residual=x, ln_weight=w32,
                                       ln_bias=_aligned(next_b.detach().float()), ln_eps=next_eps, train=True)
        ctx.save_for_backward(x, normed, w1_16, b1_32, w2_16, ln_w32, y, w32)
        ctx.eps, ctx.ln_dtypes = next_eps, (next_w.dtype, next_b.dtype)
        return y, nxt

    @staticmethod
    def backward(ctx, dy, d_next=None):
        x, normed, w1, b1, w2, ln_w, *nxt = ctx.saved_tensors
        need = ctx.needs_input_grad
        d_nxt = (None, None)
        if nxt:
            dy, *d_nxt = _through_norm(ctx, nxt[0], nxt[1], dy, d_next)
        if dy is None:
            return (None,) * 12
        dy16 = _aligned(dy.to(x.dtype))
        linear1, linear2 = need[5] or need[6], need[7] or need[8]
        if torch.is_grad_enabled():  # create_graph: the same formulas as tensor ops on the parameters, differentiable again
            with torch.autocast("cuda", enabled=False):
                lw, lb, p1, pb1, p2 = _kept_parameters(ctx)[:5]
                w1, b1, w2 = (p.to(x.dtype) for p in (p1, pb1, p2))
                u = torch.nn.functional.layer_norm(x.float(), x.shape[-1:], lw.float(), lb.float(), ctx.norm_eps).to(x.dtype)
                h = torch.nn.functional.linear(u, w1, b1)
                act, dh = torch.nn.functional.gelu(h), torch.ops.aten.gelu_backward(dy16 @ w2, h)
                dx, d_ln, d_lb = _layernorm_grad_ops(x, dh @ w1, lw, ctx.norm_eps, dy16)
                rows = lambda d, i: (_rows(d).float().t() @ _rows(i).float(), _rows(d).sum(0, dtype=torch.float32))
                grads = (*(rows(dh, u) if linear1 else (None, None)), *(rows(dy16, act) if linear2 else (None, None)), d_ln, d_lb)
        else:
            dx, *grads = PF.norm_mlp_backward(normed, dy16, x, w1, b1, w2, ln_w, ctx.norm_eps, linear1, linear2,
                                              need[0] or need[2] or need[3])
        wanted = need[5:9] + need[2:4]
        d_w1, d_b1, d_w2, d_b2, d_ln, d_lb = (g.to(t) if n else None for g, t, n in zip(grads, ctx.param_dtypes, wanted))
        return (dx, None, d_ln, d_lb, None, d_w1, d_b1, d_w2, d_b2, *d_nxt, None)


def _mlp_fused(dtype, x: torch.Tensor, layers) -> bool:
    """True where the fused bf16 MLP kernels train `layers` on rows like x's as autocast would run them."""
    lin1, act, lin2 = layers if len(layers) == 3 else (None,) * 3
    C = x.shape[-1]
    return (dtype == x.dtype == torch.bfloat16 and unhooked(layers) and _linears_served(dtype, lin1, lin2) and
            type(act) is torch.nn.GELU and unhooked(act) and act.approximate == "none" and lin1.bias is not None and
            lin2.bias is not None and lin1.in_features == lin2.out_features == C and
            PF.mlp_backward_supported(x.dtype, x.numel() // C, C, lin1.out_features))


def _next_norm(x: torch.Tensor, next_ln: torch.nn.LayerNorm | None):
    """(weight, bias, eps) of a LayerNorm that may ride in the MLP kernel's tail, else Nones."""
    if next_ln is not None and _layer_norm_served(x, next_ln) and tuple(next_ln.normalized_shape) == (x.shape[-1],):
        return next_ln.weight, next_ln.bias, next_ln.eps
    return None, None, 0.0


def norm_mlp_fused(x: torch.Tensor, ln: torch.nn.LayerNorm, layers) -> bool:
    """True where `norm_mlp_residual_of` trains y = x + Mlp(ln(x)) on rows like x's."""
    C = x.shape[-1]
    return (type(ln) is torch.nn.LayerNorm and unhooked(ln) and _layer_norm_served(x, ln) and tuple(ln.normalized_shape) == (C,) and
            _mlp_fused(compute_dtype(x), x, layers) and
            PF.norm_mlp_backward_supported(x.dtype, x.numel() // C, C, layers[0].out_features))


def norm_mlp_residual_of(x: torch.Tensor, normed: torch.Tensor, ln: torch.nn.LayerNorm, layers,
                         next_ln: torch.nn.LayerNorm | None = None):
    """(x + Mlp(ln(x)), next_ln of it or None) in training where `norm_mlp_fused`, given normed = ln(x) without a graph."""
    norm = _next_norm(x, next_ln)
    out = NormMlpResidualFunction.apply(_aligned(x), _aligned(normed), ln.weight, ln.bias, ln.eps, layers[0].weight,
                                        layers[0].bias, layers[2].weight, layers[2].bias, *norm)
    return out if norm[0] is not None else (out, None)


def mlp_residual(normed: torch.Tensor, x: torch.Tensor, layers: torch.nn.Sequential, next_ln: torch.nn.LayerNorm | None = None):
    """(x + Mlp(normed), next_ln of it or None) in training, as autocast would run it: on the fused MLP kernels where they
    serve the rows (with the LayerNorm that follows in their tail), else on `mlp`."""
    if normed.dtype == x.dtype and _mlp_fused(compute_dtype(normed), x, layers):
        norm, (lin1, _, lin2) = _next_norm(x, next_ln), layers
        out = MlpResidualFunction.apply(_aligned(normed), _aligned(x), lin1.weight, lin1.bias, lin2.weight, lin2.bias, *norm)
        return out if norm[0] is not None else (out, None)
    return mlp(normed, layers) + x, None


def norm_mlp_residual(x: torch.Tensor, ln: torch.nn.LayerNorm, layers: torch.nn.Sequential) -> torch.Tensor:
    """x + Mlp(LayerNorm(x)) in training, as autocast would run it."""
    normed, x = layer_norm_residual(x, ln)
    return mlp_residual(normed, x, layers)[0]


def layer_norm_linear(x: torch.Tensor, ln: torch.nn.LayerNorm, lin: torch.nn.Linear) -> torch.Tensor:
    """lin(ln(x)) in training (the output head), as autocast would run it: LayerNorm statistics in float32, its result
    rounded to the Linear's type."""
    dtype = compute_dtype(x)
    if x.dtype != dtype or not unhooked(ln) or not _linears_served(dtype, lin):
        return lin(ln(x))
    return linear_as_autocast(layer_norm(x, ln), lin)


def linear_as_autocast(x: torch.Tensor, lin: torch.nn.Linear) -> torch.Tensor:
    """lin(x) in training on `linear` where it serves the module, for an x in the type autocast would run it in."""
    if not _linears_served(compute_dtype(x), lin):
        return lin(x)
    if not torch.is_autocast_enabled("cuda"):
        return linear(x, lin.weight, lin.bias)
    with torch.autocast("cuda", enabled=False):
        return linear(x, lin.weight, lin.bias)


class LayerNormFunction(torch.autograd.Function):
    """LayerNorm over the last axis on the library's kernels, forward and backward, in the input's dtype (fp32 or bf16;
    statistics in fp32); x is contiguous.  The backward recomputes the statistics from the saved input."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        w32, b32 = weight.detach().float().contiguous(), bias.detach().float().contiguous()
        _, out = PF.residual_layernorm(x, ln_weight=w32, ln_bias=b32, ln_eps=eps)
        ctx.save_for_backward(x, w32)
        _keep_parameters(ctx, weight)
        ctx.eps, ctx.param_dtypes = eps, (weight.dtype, bias.dtype)
        return out

    @staticmethod
    def backward(ctx, dy):
        x, w32 = ctx.saved_tensors
        dx, dg, db = _layernorm_backward(ctx, x, dy.to(x.dtype).contiguous(), w32, ctx.eps)
        return dx, dg.to(ctx.param_dtypes[0]), db.to(ctx.param_dtypes[1]), None


class LayerNormResidualFunction(torch.autograd.Function):
    """(LayerNorm(x), x): the gradient of the second output, the residual stream going on, is added to that of the
    LayerNorm by the backward kernel instead of by a pass of its own."""

    @staticmethod
    def forward(ctx, x, weight, bias, eps):
        ctx.set_materialize_grads(False)
        return LayerNormFunction.forward(ctx, x, weight, bias, eps), x.view_as(x)

    @staticmethod
    def backward(ctx, dy, d_pass):
        if dy is None:
            return d_pass, None, None, None
        x, w32 = ctx.saved_tensors
        add = None if d_pass is None else _aligned(d_pass.to(x.dtype))
        dx, dg, db = _layernorm_backward(ctx, x, dy.to(x.dtype).contiguous(), w32, ctx.eps, add)
        return dx, dg.to(ctx.param_dtypes[0]), db.to(ctx.param_dtypes[1]), None


def _layer_norm_served(x: torch.Tensor, ln: torch.nn.LayerNorm) -> bool:
    return len(ln.normalized_shape) == 1 and ln.elementwise_affine and ln.bias is not None and PF.layernorm_supported(x)


def layer_norm_residual(x: torch.Tensor, ln: torch.nn.LayerNorm):
    """(LayerNorm(x), x) for a pre-norm block: use the second element as the residual stream."""
    if _layer_norm_served(x, ln) and x.requires_grad and torch.is_grad_enabled():
        return LayerNormResidualFunction.apply(x.contiguous(), ln.weight, ln.bias, ln.eps)
    return layer_norm(x, ln), x


def layer_norm(x: torch.Tensor, ln: torch.nn.LayerNorm) -> torch.Tensor:
    """Differentiable LayerNorm: the library's kernels where they serve the rows, the module itself otherwise."""
    if _layer_norm_served(x, ln):
        return LayerNormFunction.apply(x.contiguous(), ln.weight, ln.bias, ln.eps)
    return ln(x)
