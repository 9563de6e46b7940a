"""Backward pass of the HIP layer against autograd over the fp32 oracle (the oracle's own gradient is pinned by
finite differences in test_oracle_closed_forms.py).  Bars: fp32 gradients rtol 1e-4 with atol = 1e-4 * max|ref|
per tensor; bf16 gradients rel-L2 <= 3e-2 against the fp32 reference gradients."""
import copy
import ctypes

import numpy as np
import pytest
import torch
import torch.nn.functional as F

from oracle import torch_oracle as to
import physicsnemo_amd as pn
from physicsnemo_amd import _lib
from physicsnemo_amd import autograd as PA
from physicsnemo_amd import functional as PF
from physicsnemo_amd.transolver import Mlp
from gpu_util import announce, assert_fp32_close, assert_rel_l2, make_pair

pytestmark = pytest.mark.gpu


def _grads(module, x, probe):
    """Gradients of sum(module(x) * probe) w.r.t. x and every parameter."""
    module.zero_grad(set_to_none=True)
    x = x.clone().requires_grad_(True)
    y = module(x)
    (y.float() * probe.to(y.device)).sum().backward()
    out = {"x": x.grad}
    out.update({name: p.grad for name, p in module.named_parameters()})
    return y, out


CASES = [
    ("irregular", dict(dim=32, heads=4, dim_head=8, slice_num=8), 2, 300, None, 3),
    ("irregular", dict(dim=64, heads=2, dim_head=32, slice_num=64), 1, 1000, None, 3),
    ("irregular", dict(dim=48, heads=3, dim_head=16, slice_num=20), 3, 77, None, 3),
    ("structured2d", dict(dim=32, heads=4, dim_head=8, slice_num=8), 2, 63, (7, 9), 3),
    ("structured2d", dict(dim=16, heads=2, dim_head=8, slice_num=8), 1, 30, (5, 6), 5),
    ("structured3d", dict(dim=16, heads=2, dim_head=8, slice_num=8), 2, 60, (3, 4, 5), 3),
]


@pytest.mark.parametrize("variant,kw,B,N,grid,kernel", CASES)
def test_fp32_layer_gradients(variant, kw, B, N, grid, kernel):
    announce("fp32 backward", variant, kw, B, N, grid, kernel)
    heads = kw["heads"]
    temps = [0.3, 1.0, 2.5, 7.0][:heads] if heads <= 4 else None  # heads outside [0.5, 5] get zero temperature grad
    ref, hip = make_pair(variant, kw["dim"], heads, kw["dim_head"], kw["slice_num"], spatial=grid, kernel=kernel,
                         sharpen=2.0, temps=temps)
    ref.train(), hip.train()
    x = torch.randn(B, N, kw["dim"])
    probe = torch.randn(B, N, kw["dim"])
    y_ref, want = _grads(ref, x, probe)
    y_hip, got = _grads(hip, x.cuda(), probe)
    assert_fp32_close(y_hip, y_ref, "forward y (training path)")
    assert set(got) == set(want)
    for name in want:
        assert got[name] is not None and got[name].shape == want[name].shape, name
        assert_fp32_close(got[name], want[name], f"grad {name}", rtol=2e-4)
    if temps is not None:
        t = got["temperature"].flatten().cpu()
        assert t[0] == 0.0 and (heads < 4 or t[3] == 0.0)
        assert t[1] != 0.0


def test_slice_attention_backward_stage():
    announce("slice attention backward stage")
    B, H, S, D = 2, 3, 24, 16
    torch.manual_seed(3)
    tok = torch.randn(B, H, S, D)
    wqkv = torch.randn(3 * D, D) / D ** 0.5
    d_out = torch.randn(B, H, S, D)
    tok_r, w_r = tok.clone().requires_grad_(True), wqkv.clone().requires_grad_(True)
    q, k, v = (tok_r @ w_r.t()).chunk(3, dim=-1)
    out = torch.softmax(q @ k.transpose(-1, -2) / D ** 0.5, dim=-1) @ v
    (out * d_out).sum().backward()
    dims = PF.LayerDims(B, 100, H * D, H, D, S)
    params = {"qkv_project_weight": wqkv.cuda().contiguous()}
    d_tok, d_norm, d_w = PF.slice_attention_backward(tok.cuda(), None, d_out.cuda(), params, dims)
    assert d_norm is None
    assert_fp32_close(d_tok, tok_r.grad, "d slice_token")
    assert_fp32_close(d_w, w_r.grad, "d qkv weight")


@pytest.mark.parametrize("S,D", [(1, 8), (16, 32), (33, 16), (64, 32), (64, 64), (128, 32), (96, 40), (100, 32), (128, 64)])
@pytest.mark.parametrize("with_norm", [False, True])
def test_slice_attention_backward_tiles(S, D, with_norm):
    """The slice-attention backward over the shapes where its 32 x 32 tiles are ragged, where the S x S matrices move
    from LDS to the scratch (S = 128) and where the fma kernel takes over: against autograd in float64."""
    announce("slice attention backward", S, D, with_norm)
    B, H = 2, 2
    torch.manual_seed(S + D)
    tok, d_out = torch.randn(B, H, S, D), torch.randn(B, H, S, D)
    wqkv = torch.randn(3 * D, D) / D ** 0.5
    norm = torch.rand(B, H, S) + 0.5
    num_r = (tok.double() * norm.double()[..., None]).requires_grad_(True)
    nrm_r, w_r = norm.double().requires_grad_(True), wqkv.double().requires_grad_(True)
    tok_r = num_r / nrm_r[..., None]
    q, k, v = (tok_r @ w_r.t()).chunk(3, dim=-1)
    out = torch.softmax(q @ k.transpose(-1, -2) / D ** 0.5, dim=-1) @ v
    d_tok_r, = torch.autograd.grad((out * d_out.double()).sum(), tok_r, retain_graph=True)
    (out * d_out.double()).sum().backward()
    dims = PF.LayerDims(B, 100, H * D, H, D, S)
    if not PF.backward_supported(torch.float32, dims):
        pytest.skip("shape outside the backward kernels' range")
    params = {"qkv_project_weight": wqkv.cuda().contiguous()}
    d_num, d_norm, d_w = PF.slice_attention_backward(tok.cuda(), norm.cuda() if with_norm else None, d_out.cuda(), params,
                                                     dims)
    assert_fp32_close(d_num, num_r.grad if with_norm else d_tok_r, "d slice numerators / tokens")
    if with_norm:
        assert_fp32_close(d_norm, nrm_r.grad, "d slice norms")
    assert_fp32_close(d_w, w_r.grad, "d qkv weight")


def test_bf16_layer_gradients():
    announce("bf16 backward (autocast)")
    ref, hip = make_pair("irregular", 256, 8, 32, 64, sharpen=2.0)
    ref.train(), hip.train()
    torch.manual_seed(5)
    x = torch.randn(2, 2048, 256)
    probe = torch.randn(2, 2048, 256)
    _, want = _grads(ref, x, probe)
    hip.zero_grad(set_to_none=True)
    xc = x.cuda().requires_grad_(True)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = hip(xc)
    assert y.dtype == torch.bfloat16
    (y.float() * probe.cuda()).sum().backward()
    got = {"x": xc.grad}
    got.update({name: p.grad for name, p in hip.named_parameters()})
    for name in want:
        assert got[name].dtype == torch.float32 and torch.isfinite(got[name]).all(), name
        assert_rel_l2(got[name], want[name], f"bf16 grad {name}", tol=3e-2)


def test_model_training_step_matches_oracle():
    announce("Transolver training step fp32")
    torch.manual_seed(0)
    kw = dict(functional_dim=2, out_dim=3, embedding_dim=3, n_layers=2, n_hidden=32, n_head=4, slice_num=8, mlp_ratio=2)
    m = pn.Transolver(use_te=False, **kw).cuda().train()
    ref = to.OracleTransolver(**kw).train()
    ref.load_state_dict(m.state_dict())
    fx, emb, target = torch.randn(2, 200, 2), torch.randn(2, 200, 3), torch.randn(2, 200, 3)
    loss_ref = ((ref(fx, emb) - target) ** 2).mean()
    loss_ref.backward()
    loss = ((m(fx.cuda(), emb.cuda()) - target.cuda()) ** 2).mean()
    loss.backward()
    assert abs(float(loss.detach()) - float(loss_ref.detach())) <= 1e-4 * abs(float(loss_ref.detach()))
    want = dict(ref.named_parameters())
    for name, p in m.named_parameters():
        assert p.grad is not None, name
        assert_fp32_close(p.grad, want[name].grad, f"grad {name}", rtol=5e-4)
    # the same optimiser step on both sides leads to the same new loss
    torch.optim.SGD(m.parameters(), lr=0.01).step()
    torch.optim.SGD(ref.parameters(), lr=0.01).step()
    with torch.no_grad():
        loss2 = float(((m(fx.cuda(), emb.cuda()) - target.cuda()) ** 2).mean())
        loss2_ref = float(((ref(fx, emb) - target) ** 2).mean())
    assert abs(loss2 - loss2_ref) <= 1e-4 * abs(loss2_ref)
    assert loss2_ref >= float(loss_ref.detach()) or loss2 < float(loss.detach())


def test_gradients_reach_the_input_only_when_asked():
    announce("needs_input_grad handling")
    _, hip = make_pair("irregular", 32, 4, 8, 8)
    for p in hip.parameters():
        p.requires_grad_(False)
    x = torch.randn(1, 50, 32, device="cuda", requires_grad=True)
    hip(x).sum().backward()
    assert x.grad is not None and torch.isfinite(x.grad).all()
    assert all(p.grad is None for p in hip.parameters())


@pytest.mark.parametrize("B,N,C,S", [(2, 2048, 256, 64), (3, 1000, 128, 32), (1, 77, 128, 16), (2, 333, 256, 32),
                                     (2, 1500, 256, 128), (1, 999, 128, 128)])
def test_bf16_mfma_backward_matches_oracle_and_general_path(B, N, C, S):
    """Shapes the bf16 MFMA backward serves (ragged N, B > 1, every S <= 64): gradients against the fp32 oracle and
    against the general-kernel backward run on the same bf16 inputs."""
    announce("bf16 MFMA backward", B, N, C, S)
    from physicsnemo_amd import autograd as PA
    H = C // 32
    ref, hip = make_pair("irregular", C, H, 32, S, sharpen=2.0, temps=[0.3 + 0.4 * k for k in range(H)])
    ref.train(), hip.train()
    torch.manual_seed(9)
    x, probe = torch.randn(B, N, C), torch.randn(B, N, C)
    _, want = _grads(ref, x, probe)
    xb = x.cuda().bfloat16()
    dims = hip.layer_dims(xb)
    assert PF.mfma_backward_supported(torch.bfloat16, dims)

    def run(fn):
        hip.zero_grad(set_to_none=True)
        xc = xb.clone().requires_grad_(True)
        params = (hip.in_project_x.weight, hip.in_project_x.bias, hip.in_project_fx.weight, hip.in_project_fx.bias,
                  hip.in_project_slice.weight, hip.in_project_slice.bias, hip.temperature, hip.qkv_project.weight,
                  hip.out_linear.weight, hip.out_linear.bias)
        y = fn.apply(xc, dims, hip.kernel_params(torch.bfloat16, xc.device), *params)
        (y.float() * probe.cuda()).sum().backward()
        out = {"x": xc.grad.float()}
        out.update({name: p.grad.clone() for name, p in hip.named_parameters()})
        return out

    got = run(PA.PhysicsAttentionMfmaFunction)
    general = run(PA.PhysicsAttentionFunction)
    for name in want:
        assert torch.isfinite(got[name]).all(), name
        # d temperature is H scalars, each a sum of cancelling terms d l * logit over all points and slices; both
        # kernels keep sum_s d l = 0 per point (weights renormalised / softmax re-formed in float32), which holds it
        # to the bar of the tensor-valued gradients
        assert_rel_l2(got[name], want[name], f"MFMA bf16 grad {name} vs fp32 oracle", tol=3e-2)
        # two bf16 paths, each within 3e-2 of the oracle: their mutual distance may reach the sum for the H scalars
        assert_rel_l2(got[name], general[name], f"MFMA vs general bf16 grad {name}",
                      tol=6e-2 if name == "temperature" else 3e-2)
    t = got["temperature"].flatten().cpu()
    assert t[0] == 0.0  # 0.3 is below the clamp: no gradient


@pytest.mark.parametrize("variant,C,S,B,N,grid", [
    ("irregular", 512, 64, 2, 333, None), ("irregular", 512, 128, 1, 100, None), ("irregular", 128, 64, 1, 1, None),
    ("plus", 256, 64, 2, 1001, None), ("plus", 128, 16, 1, 63, None), ("plus", 128, 32, 3, 257, None),
    ("plus", 512, 64, 1, 96, None), ("plus", 256, 128, 1, 130, None),
    ("structured2d", 256, 64, 2, 21 * 17, (21, 17)), ("structured2d", 128, 16, 1, 33, (3, 11)),
    ("structured2d", 512, 32, 1, 40, (8, 5)), ("structured3d", 256, 128, 1, 210, (5, 6, 7)),
])
def test_bf16_training_kernels_over_variants(variant, C, S, B, N, grid):
    """Forward and backward of the bf16 training calls where their tiles, head groups and table forms change: every
    parameter tensor and the input gradient against the fp32 oracle (bf16 data: 3e-2; the few scalars, sums of cancelling
    terms, only have to be finite)."""
    announce("bf16 training kernels", variant, C, S, B, N, grid)
    H = C // 32
    torch.manual_seed(S + N)
    plus = variant == "plus"
    if plus:
        ref = to.OraclePhysicsAttentionIrregularMesh(C, heads=H, dim_head=32, slice_num=S, plus=True)
        hip = pn.PhysicsAttentionIrregularMesh(C, heads=H, dim_head=32, slice_num=S, use_te=False, plus=True)
        hip.load_state_dict(ref.state_dict())
        hip = hip.cuda()
    else:
        ref, hip = make_pair(variant, C, H, 32, S, spatial=grid, sharpen=2.0)
    ref.train(), hip.train()
    xb = torch.randn(B, N, C).bfloat16()
    probe = torch.randn(B, N, C).bfloat16()
    u = torch.rand(B, N, H, S).bfloat16()
    assert PF.layer_train_supported(torch.bfloat16, hip.layer_dims(xb.cuda()), plus)

    def run(m, x, probe, u):
        x = x.clone().requires_grad_(True)
        y = m.forward_with_noise(x, u) if plus else m(x)
        y.backward(probe)
        return y.detach(), {"x": x.grad, **{n: p.grad for n, p in m.named_parameters()}}

    y_ref, want = run(ref, xb.float(), probe.float(), u.float())
    y, got = run(hip, xb.cuda(), probe.cuda(), u.cuda())
    assert_rel_l2(y, y_ref, "y (training forward)", tol=1e-2)
    for name in want:
        assert torch.isfinite(got[name]).all(), name
        if want[name].numel() >= 32 and N > 1:
            assert_rel_l2(got[name], want[name], f"grad {name}", tol=3e-2)


@pytest.mark.parametrize("variant,C,S,B,N,grid", [
    ("irregular", 512, 128, 1, 2048, None), ("irregular", 512, 32, 2, 1001, None), ("plus", 256, 64, 1, 4003, None),
    ("plus", 128, 16, 2, 2001, None), ("structured2d", 256, 64, 1, 1200, (30, 40)), ("structured2d", 128, 32, 2, 660, (20, 33)),
])
def test_bf16_training_gradients_keep_float32_tables(variant, C, S, B, N, grid):
    """Layers whose backward multiplies with float32 tables (slice weights, attended tokens, d num): every gradient, the
    temperature's among them, against float64 at large weights that bf16 holds.  A chain has at most six independent
    bf16 roundings of per-point values (x_mid, fx_mid, d out_x, d z, d x_mid, the result: 2^-9 / sqrt(3) = 1.1e-3 of a value
    on the average each, 2.8e-3 together); 5e-3 leaves room for the cancellation in sums over the points, and gradients
    of a few elements (temperature, last bias of proj_temperature) get 1e-2.  Tables rounded to bf16 put one and the same error into every point, which
    the sums do not average: 0.7e-2 to 1.6e-2 at 512 channels."""
    announce("float32 tables in bf16 training", variant, C, S, B, N, grid)
    H = C // 32
    plus = variant == "plus"
    if plus:
        torch.manual_seed(0)
        ref = to.OraclePhysicsAttentionIrregularMesh(C, heads=H, dim_head=32, slice_num=S, plus=True)
        hip = pn.PhysicsAttentionIrregularMesh(C, heads=H, dim_head=32, slice_num=S, use_te=False, plus=True).cuda()
    else:
        ref, hip = make_pair(variant, C, H, 32, S, spatial=grid)
    with torch.no_grad():
        for name, p in ref.named_parameters():
            if name == "temperature":
                p.copy_(0.6 + 0.8 * torch.rand_like(p))
            elif name.split(".")[0] in ("in_project_x", "in_project_fx", "out_linear") and p.ndim > 1:
                p.copy_(p.bfloat16().float())
            elif name.endswith("bias"):
                p.add_(0.1 * torch.randn_like(p))
    hip.load_state_dict(ref.state_dict())
    ref, hip = ref.double().train(), hip.train()
    x, dy, u = torch.randn(B, N, C).bfloat16(), torch.randn(B, N, C).bfloat16(), torch.rand(B, N, H, S).bfloat16()
    assert PF.layer_train_supported(torch.bfloat16, hip.layer_dims(x.cuda()), plus)

    def run(m, x, dy, u):
        x = x.clone().requires_grad_(True)
        y = m.forward_with_noise(x, u) if plus else m(x)
        y.backward(dy)
        return {"y": y.detach(), "x": x.grad, **{n: p.grad for n, p in m.named_parameters()}}

    want, got = run(ref, x.double(), dy.double(), u.double()), run(hip, x.cuda(), dy.cuda(), u.cuda())
    for name in want:
        assert_rel_l2(got[name], want[name], name, tol=1e-2 if want[name].numel() < 16 else 5e-3)


@pytest.mark.parametrize("rows", [1, 33, 2015])
@pytest.mark.parametrize("ca,cb", [(256, 256), (512, 128), (256, 16)])
def test_weight_gradient_with_an_infinite_last_row(rows, ca, cb):
    """An infinity in the last row of a ragged count stays one in the column it belongs to: the rows that only fill the last
    tile do not turn it into a NaN, nor do they reach other columns."""
    announce("infinite last row", rows, ca, cb)
    a, b = (1 + torch.rand(rows, c, device="cuda").bfloat16() for c in (ca, cb))
    for inf_in_a in (False, True):
        x, y = a.clone(), b.clone()
        (x if inf_in_a else y)[-1, 3] = float("inf")
        got, sums = PF.cols_gemm(x, y, col_sums=True)
        want = torch.zeros(ca, cb, dtype=torch.bool, device="cuda")
        (want[3] if inf_in_a else want[:, 3]).fill_(True)
        assert not got.isnan().any() and torch.equal(got.isinf(), want)
        assert not sums.isnan().any() and sums.isinf().sum() == int(inf_in_a)


@pytest.mark.parametrize("C,S,B,N", [(256, 64, 5, 70), (256, 64, 130, 33), (128, 16, 300, 20), (512, 128, 37, 31),
                                     (256, 32, 9, 2100)])
def test_many_clouds_in_one_training_batch(C, S, B, N):
    """The gradients that come from sums per batch element where those go through in groups, partly filled ones among them,
    and d W_out is formed in parts: against float64.  The workspace holds one group's sums."""
    announce("many clouds", C, S, B, N)
    H = C // 32
    ref, hip = make_pair("irregular", C, H, 32, S)
    with torch.no_grad():
        for m in (ref, hip):
            for w in (m.in_project_x.weight, m.in_project_fx.weight, m.out_linear.weight):
                w.copy_(w.bfloat16().float())
    ref, hip = ref.double().cuda().train(), hip.train()
    x, dy = torch.randn(2, B, N, C, device="cuda").bfloat16()

    def run(m, x, dy):
        x = x.clone().requires_grad_(True)
        m(x).backward(dy)
        return {"x": x.grad, **{n: p.grad for n, p in m.named_parameters()}}

    want, got = run(ref, x.double(), dy.double()), run(hip, x, dy)
    # d W_out = dy^T out_x: the weights' bf16 rounding averages out over the points, as for d W_qkv behind the tokens
    for name in ("out_linear.weight", "out_linear.bias", "qkv_project.weight"):
        assert_rel_l2(got[name], want[name], name, tol=2e-3)
    for name in ("x", "in_project_x.weight", "in_project_fx.weight", "in_project_slice.weight"):
        assert_rel_l2(got[name], want[name], name, tol=2e-2)
    dims = hip.layer_dims(x)
    floats = _lib.load().pa_output_backward_workspace_bytes(ctypes.byref(dims.c())) / 4
    assert floats <= 2 * 256 * 256 * 256 + B * C * 256 + 33 * C * C


def test_mfma_deslice_natural_layout():
    announce("MFMA deslice to natural layout")
    ref, hip = make_pair("irregular", 256, 8, 32, 64, sharpen=2.0)
    x = torch.randn(2, 500, 256)
    xb = x.cuda().bfloat16()
    dims = hip.layer_dims(xb)
    with torch.no_grad():
        st = PF.MfmaStages(hip.kernel_params(torch.bfloat16, xb.device), dims, xb.device)
        st.pack_params()
        st.project_softmax_reduce(xb)
        st.combine_attention()
        out_x = st.deslice()
        stages = ref.stages(x)
        want = torch.einsum("bths,bhsd->bthd", stages["w"], stages["tok_out"]).reshape(2, 500, 256)
        assert_rel_l2(out_x, want, "out_x")
        # packed and natural outputs of the row GEMM agree: the packed copy feeds the slice sum, compare through it
        w = hip.out_linear.weight.detach().bfloat16().t().contiguous()  # any (256, 256) weight
        nat, pack = st.rows_gemm_packed(xb, w, None)
        assert_rel_l2(nat, x @ w.float().cpu().t(), "natural GEMM output")
        sums = st.slice_weighted_sum(pack)
        want_sums = torch.einsum("bnhs,bnhd->bhsd", stages["w"], (x @ w.float().cpu().t()).reshape(2, 500, 8, 32))
        assert_rel_l2(sums[..., :32], want_sums, "slice sums of the packed GEMM output")
        assert_rel_l2(sums[..., 32], stages["w"].sum(1), "slice counts")


@pytest.mark.parametrize("rows,ca,cb", [(5000, 64, 32), (1000, 256, 256), (333, 512, 256), (31, 32, 32), (70000, 256, 128)])
def test_cols_gemm_weight_gradient_product(rows, ca, cb):
    announce("cols_gemm", rows, ca, cb)
    torch.manual_seed(rows)
    a = torch.randn(rows, ca, device="cuda").bfloat16()
    b = torch.randn(rows, cb, device="cuda").bfloat16()
    assert PF.cols_gemm_supported(a, b)
    got, sums = PF.cols_gemm(a, b, col_sums=True)
    assert_fp32_close(sums, a.double().sum(0).float(), "column sums of a", rtol=1e-4)
    want = a.double().t() @ b.double()  # exact products of the bf16 inputs; the kernel accumulates them in fp32
    assert got.shape == (ca, cb) and got.dtype == torch.float32
    assert_fp32_close(got, want.float(), "a^T b", rtol=1e-4)
    assert torch.equal(got, PF.cols_gemm(a, b))  # fixed summation order


@pytest.mark.parametrize("rows,ca,cb", [(5000, 64, 32), (4099, 256, 256), (8192, 512, 132), (70001, 4, 260), (300000, 128, 256)])
def test_cols_gemm_float32(rows, ca, cb):
    announce("cols_gemm float32", rows, ca, cb)
    torch.manual_seed(rows)
    a = torch.randn(rows, ca, device="cuda") + 0.25
    b = torch.randn(rows, cb, device="cuda")
    assert PF.cols_gemm_supported(a, b)
    got, sums = PF.cols_gemm(a, b, col_sums=True)
    assert_fp32_close(sums, a.double().sum(0).float(), "column sums of a", rtol=1e-4)
    want = a.double().t() @ b.double()
    assert got.shape == (ca, cb) and got.dtype == torch.float32
    assert_fp32_close(got, want.float(), "a^T b", rtol=1e-4)
    assert torch.equal(got, PF.cols_gemm(a, b))  # fixed summation order


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("rows,ca,cb", [
    (1, 256, 256), (33, 128, 128), (4097, 1024, 256), (2500, 256, 1024), (100001, 512, 288), (777, 160, 416),  # tile kernels
    (5, 512, 5), (100003, 512, 7), (3001, 4, 256), (64, 1, 64), (9000, 260, 16), (129, 16, 300),               # one narrow side
])
def test_weight_gradient_shapes(dtype, rows, ca, cb):
    """Row counts around the 32-row stages and the chunks, widths around the 256-column blocks, both narrow sides:
    against float64, to the rounding of an fp32 sum of `rows` products (about sqrt(rows) 6e-8 of the rms entry)."""
    announce("weight gradient", dtype, rows, ca, cb)
    torch.manual_seed(rows + ca)
    a = torch.randn(rows, ca, device="cuda").to(dtype)
    b = (torch.randn(rows, cb, device="cuda") + 0.1).to(dtype)
    if not PF.cols_gemm_supported(a, b):
        pytest.skip("width pair left to the GEMM library")
    got, sums = PF.cols_gemm(a, b, col_sums=True)
    assert_fp32_close(got, (a.double().t() @ b.double()).float(), "a^T b", rtol=1e-4)
    assert_fp32_close(sums, a.double().sum(0).float(), "column sums", rtol=1e-4)
    assert torch.equal(got, PF.cols_gemm(a, b))


@pytest.mark.parametrize("rows,ca,cb", [
    (30011, 1024, 256), (9000, 512, 256), (12000, 1024, 256), (70001, 256, 256),  # few / many partials, large / small result
    (4100, 256, 3), (1000, 3, 20), (65, 5, 16),                                   # results of 4 k and of other numbers of values
])
def test_totals_of_partial_products(rows, ca, cb):
    """The splits of a total among a workgroup's rows of lanes.  Inputs are small whole numbers, so that every float32 sum
    is exact and the results equal float64's to the bit."""
    announce("totals of partial products", rows, ca, cb)
    torch.manual_seed(rows)
    a, b = (torch.randint(-3, 4, (rows, c), device="cuda").bfloat16() for c in (ca, cb))  # |sums| <= 9 rows < 2^24
    got, sums = PF.cols_gemm(a, b, col_sums=True)
    assert torch.equal(got, (a.double().t() @ b.double()).float())
    assert torch.equal(sums, a.double().sum(0).float())


@pytest.mark.parametrize("rows,ca,cb", [(30011, 256, 64), (32768, 1024, 256), (50000, 512, 256)])
def test_totals_add_their_parts_in_halves(rows, ca, cb):
    """Sums of random values over the rows, in up to 32 parts: 6.1e-8 to 6.5e-8 off float64 with halves added to halves, 1.0e-7 to
    1.1e-7 with one part after the other, whose roundings a sum of that many values of one size adds up (7.0e-8 to 7.5e-8: eight
    parts)."""
    announce("totals in halves", rows, ca, cb)
    square = 0.0
    for seed in range(6):
        torch.manual_seed(seed)
        a, b = (torch.randn(rows, c, device="cuda").bfloat16() for c in (ca, cb))
        want = a.double().sum(0)
        square += ((PF.cols_gemm(a, b, col_sums=True)[1] - want).norm() / want.norm()).item() ** 2 / 6
    assert square ** 0.5 <= 7.5e-8, square ** 0.5


@pytest.mark.parametrize("dtype,C,O", [(torch.bfloat16, 256, 512), (torch.bfloat16, 128, 128), (torch.float32, 128, 256),
                                       (torch.float32, 36, 20)])
@pytest.mark.parametrize("grid,k", [((13, 9), 3), ((40, 33), 5), ((4, 6, 5), 3), ((1, 50), 3)])
def test_conv_weight_gradient(dtype, C, O, grid, k):
    """The convolution form (neighbours gathered per tap, zero outside the grid) against torch's convolution backward."""
    announce("conv weight gradient", dtype, C, O, grid, k)
    torch.manual_seed(C + k)
    B, N = 2, int(np.prod(grid))
    g, x = torch.randn(B, N, O, device="cuda").to(dtype), torch.randn(B, N, C, device="cuda").to(dtype)
    dims = PF.LayerDims(B, N, C, 4, 32, 32, grid[0], grid[1], k, grid[2] if len(grid) == 3 else 0, 1)
    assert PF.cols_gemm_supported(g, x, dims)
    dw, db = PF.cols_gemm(g, x, col_sums=True, grid=dims)
    w = torch.zeros(O, C, *(k,) * len(grid), dtype=torch.float64, requires_grad=True)
    conv = torch.nn.functional.conv2d if len(grid) == 2 else torch.nn.functional.conv3d
    y = conv(x.double().cpu().transpose(1, 2).reshape(B, C, *grid), w, padding=k // 2)
    y.backward(g.double().cpu().transpose(1, 2).reshape(B, O, *grid))
    assert_fp32_close(dw, w.grad, "d weight")
    assert_fp32_close(db, g.double().sum((0, 1)), "d bias")


def test_bf16_model_training_step_runs_the_mfma_backward():
    announce("Transolver training step, bf16 autocast, MFMA backward inside the blocks")
    torch.manual_seed(1)
    kw = dict(functional_dim=3, out_dim=2, embedding_dim=2, n_layers=2, n_hidden=128, n_head=4, slice_num=32, mlp_ratio=2)
    m = pn.Transolver(use_te=False, **kw).cuda().train()
    ref = to.OracleTransolver(**kw).train()
    ref.load_state_dict(m.state_dict())
    fx, emb, target = torch.randn(2, 700, 3), torch.randn(2, 700, 2), torch.randn(2, 700, 2)
    ((ref(fx, emb) - target) ** 2).mean().backward()
    with torch.autocast("cuda", dtype=torch.bfloat16):
        out = m(fx.cuda(), emb.cuda())
    ((out.float() - target.cuda()) ** 2).mean().backward()
    want = dict(ref.named_parameters())
    for name, p in m.named_parameters():
        assert p.grad is not None and torch.isfinite(p.grad).all(), name
        if "temperature" in name or want[name].grad.abs().max() < 1e-6:
            continue
        assert_rel_l2(p.grad, want[name].grad, f"bf16 model grad {name}", tol=8e-2)


def test_mfma_backward_at_scale_agrees_with_general_path():
    """200 000 points (more than any CPU-oracle case): the MFMA backward and the general backward, two independent
    implementations of the same gradient, agree on the same bf16 inputs; the input gradient is finite everywhere."""
    announce("MFMA vs general backward at 200k points")
    from physicsnemo_amd import autograd as PA
    _, hip = make_pair("irregular", 256, 8, 32, 64, sharpen=2.0)
    hip.train()
    torch.manual_seed(2)
    N = 200_000
    xb = torch.randn(1, N, 256, device="cuda").bfloat16()
    probe = torch.randn(1, N, 256, device="cuda").bfloat16()
    dims = hip.layer_dims(xb)
    params = (hip.in_project_x.weight, hip.in_project_x.bias, hip.in_project_fx.weight, hip.in_project_fx.bias,
              hip.in_project_slice.weight, hip.in_project_slice.bias, hip.temperature, hip.qkv_project.weight,
              hip.out_linear.weight, hip.out_linear.bias)
    res = []
    for fn in (PA.PhysicsAttentionMfmaFunction, PA.PhysicsAttentionFunction):
        hip.zero_grad(set_to_none=True)
        xc = xb.clone().requires_grad_(True)
        y = fn.apply(xc, dims, hip.kernel_params(torch.bfloat16, xc.device), *params)
        y.backward(probe)
        g = {"x": xc.grad.float()}
        g.update({n: p.grad.clone() for n, p in hip.named_parameters()})
        res.append(g)
    assert torch.isfinite(res[0]["x"]).all()
    for name in res[0]:
        if name != "temperature":
            assert_rel_l2(res[0][name], res[1][name], f"grad {name}", tol=3e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,C", [(1000, 256), (37, 48), (4096, 512), (300, 1024)])
def test_layernorm_and_linear_autograd_functions(dtype, rows, C):
    announce("LayerNormFunction / LinearFunction", dtype, rows, C)
    from physicsnemo_amd import autograd as PA
    torch.manual_seed(rows)
    ln = torch.nn.LayerNorm(C)
    with torch.no_grad():
        ln.weight.uniform_(0.5, 1.5)
        ln.bias.uniform_(-0.5, 0.5)
    x, probe = torch.randn(2, rows, C), torch.randn(2, rows, C)
    xr = x.to(dtype).float().clone().requires_grad_(True)  # reference: fp32 arithmetic on the same (rounded) input
    (ln(xr) * probe).sum().backward()
    want = (xr.grad, ln.weight.grad.clone(), ln.bias.grad.clone())
    ln.zero_grad()
    lng = ln.cuda()
    xg = x.detach().to(dtype).cuda().requires_grad_(True)
    y = PA.layer_norm(xg, lng)
    assert y.dtype == dtype and y.grad_fn is not None
    (y.float() * probe.cuda()).sum().backward()
    got = (xg.grad, lng.weight.grad, lng.bias.grad)
    for name, g, w in zip(("dx", "d gamma", "d beta"), got, want):
        if dtype == torch.float32:
            assert_fp32_close(g, w, name, rtol=2e-4)
        else:
            assert_rel_l2(g, w, name, tol=1e-2)
    if dtype == torch.bfloat16:
        lin = torch.nn.Linear(C, 256)
        xr = x.detach().bfloat16().float().requires_grad_(True)
        p2 = torch.randn(2, rows, 256)
        (torch.nn.functional.linear(xr, lin.weight.bfloat16().float(), lin.bias) * p2).sum().backward()
        wx = xr.grad
        lin.zero_grad(set_to_none=True)  # the reference pass above left gradients on the parameters
        lin = lin.cuda()
        xg = x.detach().bfloat16().cuda().requires_grad_(True)
        out = PA.linear(xg, lin.weight, lin.bias)
        (out.float() * p2.cuda()).sum().backward()
        assert lin.weight.grad.dtype == torch.float32
        assert_rel_l2(xg.grad, wx, "linear dx", tol=1e-2)
        ref_dw = (p2.bfloat16().float().reshape(-1, 256).t() @ x.bfloat16().float().reshape(-1, C))
        assert_rel_l2(lin.weight.grad, ref_dw, "linear dW", tol=1e-2)
        assert_rel_l2(lin.bias.grad, p2.bfloat16().float().reshape(-1, 256).sum(0), "linear db", tol=1e-2)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,C", [(1, 8), (7, 16), (1001, 64), (300, 96), (4099, 256), (63, 520), (130, 1024)])
def test_layernorm_row_groups(dtype, rows, C):
    """The row kernels where the lanes sharing a row change (4 .. 64 and several units per lane) and rows run out inside a
    wave: forward with a residual, backward with a gradient past the LayerNorm, against float64."""
    announce("layernorm row groups", dtype, rows, C)
    torch.manual_seed(rows + C)
    y, res, dy, add = (torch.randn(rows, C, device="cuda").to(dtype) for _ in range(4))
    gam, bet = torch.randn(C, device="cuda"), torch.randn(C, device="cuda")
    fx, out = PF.residual_layernorm(y.clone(), residual=res, ln_weight=gam, ln_bias=bet)
    want_fx = (y.double() + res.double()).to(dtype)
    assert torch.equal(fx, (y.float() + res.float()).to(dtype))
    x = want_fx.double().requires_grad_(True)
    g64, b64 = gam.double().requires_grad_(True), bet.double().requires_grad_(True)
    ln = torch.nn.functional.layer_norm(x, (C,), g64, b64)
    ln.backward(dy.double())
    dx, dg, db = PF.layernorm_backward(want_fx, dy, gam, add=add)
    # bf16 results carry one rounding (2^-9 of the value), fp32 ones a few of the row sums' 2^-24
    tol = 4e-3 if dtype == torch.bfloat16 else 1e-6
    assert_rel_l2(out, ln.detach(), "LayerNorm", tol=tol)
    assert_rel_l2(dx, x.grad + add.double(), "dx + add", tol=tol)
    assert_rel_l2(dg, g64.grad, "d gamma", tol=1e-5)
    assert_rel_l2(db, b64.grad, "d beta", tol=1e-5)


@pytest.mark.parametrize("dtype,rows,C", [(torch.bfloat16, 1, 256), (torch.bfloat16, 2001, 256), (torch.float32, 7, 32),
                                          (torch.float32, 1003, 64), (torch.bfloat16, 3, 40)])
def test_layernorm_backward_without_eps(dtype, rows, C):
    """eps = 0 with rows that do not fill the last wave: the rows that are not there add nothing to d gamma."""
    announce("layernorm, eps 0", dtype, rows, C)
    x, dy = (torch.randn(rows, C, device="cuda").to(dtype) for _ in range(2))
    gam = torch.randn(C, device="cuda")
    x64, g64 = x.double().requires_grad_(True), gam.double().requires_grad_(True)
    b64 = torch.zeros_like(g64, requires_grad=True)
    torch.nn.functional.layer_norm(x64, (C,), g64, b64, eps=0.0).backward(dy.double())
    got = PF.layernorm_backward(x, dy, gam, ln_eps=0.0)
    # as with an eps: one rounding of dx to its type, float32 sums
    for g, want, tol in zip(got, (x64.grad, g64.grad, b64.grad), (4e-3 if dtype == torch.bfloat16 else 1e-6, 1e-5, 1e-5)):
        assert torch.isfinite(g).all()
        assert_rel_l2(g, want, "dx, d gamma, d beta", tol=tol)


@pytest.mark.parametrize("C,S,B,N", [(256, 64, 2, 333), (128, 16, 1, 63), (128, 128, 2, 100), (256, 32, 1, 32)])
def test_point_stages_of_the_bf16_backward_agree(C, S, B, N):
    """The stage that reads the stored slice weights and leaves d z, and the one that forms the weights again and sums
    d W_slice: the same gradients."""
    announce("point stages", C, S, B, N)
    torch.manual_seed(S)
    _, hip = make_pair("irregular", C, C // 32, 32, S)
    x, g = torch.randn(2, B, N, C, device="cuda").bfloat16()
    dims, kp = hip.layer_dims(x), hip.kernel_params(torch.bfloat16, x.device)
    st = PF.MfmaStages(kp, dims, x.device)
    st.pack_params()
    st.project_softmax(x)
    st.slice_reduce()
    st.combine_attention()
    x_mid, fx_mid = PF.project_inputs(x, kp, dims)
    d_num = torch.randn(B, dims.H, S, 32, device="cuda")
    d_norm = torch.randn(B, dims.H, S, device="cuda")
    d_proj, d_z, d_temp = st.slice_softmax_backward(x_mid, fx_mid, g, d_num, d_norm)
    want, d_ws, d_bs, want_temp = PF.point_backward(x_mid, fx_mid, g, st.tok_out, d_num, d_norm, kp, dims)
    # one side reads weights rounded to bf16 (2^-9 of each), both round d z and the result to it
    assert_rel_l2(d_proj, want, "d x_mid, d fx_mid", tol=6e-3)
    rows = d_z.float().reshape(-1, S)
    assert_rel_l2(rows.t() @ x_mid.float().reshape(-1, 32), d_ws, "d W_slice from d z", tol=1e-2)
    assert_rel_l2(d_temp, want_temp, "d temperature", tol=3e-2)


@pytest.mark.parametrize("C,S,grid", [(256, 64, (20, 33)), (128, 16, (9, 7)), (512, 128, (16, 20)), (256, 32, (8, 4))])
def test_point_backward_multiplies_float32_gradients(C, S, grid):
    """d x_mid = d z W_slice of the structured layers from given rows: d z does not lose bits on its way into the product, so
    the error against float64 is the rounding of the result alone (bf16: 1.7e-3 of a value in the mean square); d z rounded
    to bf16 first adds as much again, and more where its terms cancel."""
    announce("point backward, float32 d z", C, S, grid)
    torch.manual_seed(S)
    _, hip = make_pair("structured2d", C, C // 32, 32, S, spatial=grid, sharpen=2.0)
    x = torch.zeros(1, grid[0] * grid[1], C, device="cuda", dtype=torch.bfloat16)
    dims, kp = hip.layer_dims(x), hip.kernel_params(torch.bfloat16, x.device)
    N, H = dims.N, dims.H
    x_mid, fx_mid, g = torch.randn(3, 1, N, C, device="cuda").bfloat16()
    tok, d_num = torch.randn(2, 1, H, S, 32, device="cuda")
    d_norm = torch.randn(1, H, S, device="cuda")
    d_proj, *_ = PF.point_backward(x_mid, fx_mid, g, tok, d_num, d_norm, kp, dims)
    heads = lambda t: t.double().view(N, H, 32)
    ws, bs = kp["in_project_slice_weight"].double().view(S, 32), kp["in_project_slice_bias"].double()
    temp = kp["temperature"].double().clamp(0.5, 5.0).view(1, H, 1)
    w = torch.softmax((heads(x_mid) @ ws.t() + bs) / temp, -1)
    dw = (torch.einsum("nhd,hsd->nhs", heads(g), tok[0].double()) +
          torch.einsum("nhd,hsd->nhs", heads(fx_mid), d_num[0].double()) + d_norm.double())
    dz = w / temp * (dw - (w * dw).sum(-1, keepdim=True))
    assert_rel_l2(d_proj[0, :, :C].reshape(N, H, 32), dz @ ws, "d x_mid", tol=1.8e-3)


@pytest.mark.parametrize("dtype,rows,C", [(torch.bfloat16, 1003, 256), (torch.float32, 31, 64)])
def test_layernorm_backward_partial_sums(dtype, rows, C):
    """pa_layernorm_backward leaves the groups' shares of d gamma and d beta to the caller; their sum and dx are those of
    the call that adds them up."""
    announce("layernorm partial sums", dtype, rows, C)
    x, dy = (torch.randn(rows, C, device="cuda").to(dtype) for _ in range(2))
    gam, dx = torch.randn(C, device="cuda"), torch.empty_like(x)
    lib = _lib.load()
    partials = torch.empty(lib.pa_layernorm_backward_groups(rows), 2, C, device="cuda")
    _lib.check(lib.pa_layernorm_backward(_lib.dtype_code(dtype), rows, C, x.data_ptr(), dy.data_ptr(), gam.data_ptr(), 1e-5,
                                         dx.data_ptr(), partials.data_ptr(), _lib.current_stream_ptr(x.device)), "call")
    want_dx, dg, db = PF.layernorm_backward(x, dy, gam)
    assert torch.equal(dx, want_dx)
    for got, want in zip(partials.sum(0), (dg, db)):  # float32 sums in another order
        assert_rel_l2(got, want, "d gamma, d beta", tol=1e-6)


@pytest.mark.parametrize("grid,C,O,B,k", [((3, 5), 64, 256, 2, 3), ((16, 17), 256, 256, 1, 3), ((9, 30), 128, 512, 3, 5),
                                          ((4, 5, 7), 64, 256, 2, 3), ((33, 40), 512, 256, 1, 3)])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_convolution_as_implicit_gemm(grid, C, O, B, k, dtype):
    """The ring-buffered convolution at partial row blocks, one and several channel blocks per tap, 2-D and 3-D,
    against float64."""
    announce("conv gemm", grid, C, O, B, k, dtype)
    torch.manual_seed(C + O)
    N = int(np.prod(grid))
    dims = PF.LayerDims(B, N, C, O // 32, 32, 32, grid[0], grid[1], k, grid[2] if len(grid) == 3 else 0, 1)
    x = torch.randn(B, N, C, device="cuda").to(dtype)
    w = (torch.randn(O, C, *(k,) * len(grid), device="cuda") / (C * k ** len(grid)) ** 0.5).to(dtype)
    bias = torch.randn(O, device="cuda")
    got = PF.rows_gemm(x, w.movedim(1, -1).contiguous(), bias, dims, C, O)
    conv = torch.nn.functional.conv2d if len(grid) == 2 else torch.nn.functional.conv3d
    want = conv(x.double().transpose(1, 2).reshape(B, C, *grid).cpu(), w.double().cpu(), bias.double().cpu(), padding=k // 2)
    # one bf16 rounding of the result: at most 2^-9 of each value, 2^-9 / sqrt(3) on the average; float32: the sums' own
    # rounding, 2^-24 sqrt(terms) at 4 608 terms
    assert_rel_l2(got, want.reshape(B, O, N).transpose(1, 2), "conv", tol=2e-3 if dtype == torch.bfloat16 else 4e-6)


@pytest.mark.parametrize("rows,F", [(1, 64), (255, 128), (257, 1024), (2000, 192), (70_001, 256)])
def test_mlp_residual_block(rows, F):
    """x + Mlp(LayerNorm(x)) of a bf16 block, forward and all gradients, at partial row blocks, with the hidden units
    split between workgroups and not, and with more items than workgroups, against float64."""
    announce("mlp residual", rows, F)
    torch.manual_seed(rows)
    C = 256
    ln = torch.nn.LayerNorm(C).cuda()
    layers = torch.nn.Sequential(torch.nn.Linear(C, F), torch.nn.GELU(), torch.nn.Linear(F, C)).cuda()
    with torch.no_grad():
        ln.weight.add_(0.3 * torch.randn_like(ln.weight))
        for lin in (layers[0], layers[2]):
            lin.weight.copy_(lin.weight.bfloat16().float())
    x = torch.randn(rows, C, device="cuda").bfloat16().requires_grad_(True)
    dy = torch.randn(rows, C, device="cuda").bfloat16()
    assert PF.mlp_backward_supported(x.dtype, rows, C, F)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        y = PA.norm_mlp_residual(x, ln, layers)
    y.backward(dy)
    import copy
    ln64, layers64 = copy.deepcopy(ln).double(), copy.deepcopy(layers).double()
    ln64.zero_grad(), layers64.zero_grad()
    x64 = x.detach().double().requires_grad_(True)
    y64 = x64 + layers64(ln64(x64))
    y64.backward(dy.double())
    # every chain carries at most four bf16 roundings (LayerNorm, hidden layer or its gradient, result, sum): 2^-9 each
    # at most, 2^-9 / sqrt(3) on the average
    assert_rel_l2(y.detach(), y64.detach(), "y", tol=4e-3)
    assert_rel_l2(x.grad, x64.grad, "dx", tol=5e-3)
    for (name, p), q in zip(list(ln.named_parameters()) + list(layers.named_parameters()),
                            list(ln64.parameters()) + list(layers64.parameters())):
        assert p.grad.dtype == torch.float32
        assert_rel_l2(p.grad, q.grad, "d " + name, tol=6e-3)
    # create_graph takes the same formulas as tensor ops
    (gx,) = torch.autograd.grad(PA.norm_mlp_residual(x, ln.bfloat16(), layers.bfloat16()), x, dy, create_graph=True)
    assert_rel_l2(gx.detach(), x64.grad, "dx, create_graph", tol=1e-2)


def test_gelu_of_the_training_mlp_keeps_its_tail():
    """The hidden layer at known values over [-9, 9]: GELU and its derivative, forward and backward, are the exact ones
    rounded to bf16 once (2^-8 of a value at most), far into the lower tail; a fit that is good to 2.6e-5 absolutely is off by
    a fifth at -4."""
    announce("GELU of the training MLP")
    C = F = 256
    h = torch.linspace(-9, 9, F, device="cuda")
    rows = 300
    u = torch.randn(rows, C, device="cuda").bfloat16()
    w1, eye = torch.zeros(F, C, device="cuda", dtype=torch.bfloat16), torch.eye(C, F, device="cuda").bfloat16()
    zero = torch.zeros(C, device="cuda")
    h64 = h.double().requires_grad_(True)
    want = h64 * 0.5 * torch.erfc(-h64 / 2 ** 0.5)  # erfc keeps the relative accuracy of the tail
    (slope,) = torch.autograd.grad(want.sum(), h64)
    want = want.detach()
    residual = torch.zeros(rows, C, device="cuda", dtype=torch.bfloat16)
    y = PF.mlp_forward_packed(u, PF.mlp_pack(w1, eye), h, zero, residual=residual, train=True)
    act, dh = PF.mlp_backward(u, torch.ones(rows, C, device="cuda", dtype=torch.bfloat16), w1, h, eye)
    for got, exact, slack in ((y, want, 0.0), (act, want, 0.0), (dh, slope, 1.1e-6)):  # the slope passes through zero
        err = (got.double() - exact).abs()
        # beside the rounding: the fit's 2e-6 and the exponent's x^2 2^-24 of a value; 1 - Phi is formed in float32
        assert (err <= 2.0 ** -8 * 1.01 * exact.abs() + slack).all(), (err / exact.abs()).max()


@pytest.mark.parametrize("next_norm", [False, True])
def test_mlp_residual_block_differentiates_twice(next_norm):
    """Gradients of a function of the gradient of a bf16 block's MLP, by its input and every parameter of the Linears and of
    the LayerNorms before and behind, with float32 and with bf16 parameters, against float64.  A parameter that changed
    between the passes is refused there and only there."""
    announce("mlp residual twice", next_norm)
    torch.manual_seed(0)
    rows, C, F = 300, 256, 128
    ln, after = torch.nn.LayerNorm(C).cuda(), torch.nn.LayerNorm(C).cuda()
    layers = torch.nn.Sequential(torch.nn.Linear(C, F), torch.nn.GELU(), torch.nn.Linear(F, C)).cuda()
    modules = [ln, layers] + ([after] if next_norm else [])
    with torch.no_grad():
        for m in modules:
            for p in m.parameters():
                p.copy_((p + 0.1 * torch.randn_like(p)).bfloat16().float())
    x, dy, dn = (torch.randn(rows, C, device="cuda").bfloat16() for _ in range(3))

    def second(mods, x, call):
        x = x.detach().requires_grad_(True)
        params = [p for m in mods for p in m.parameters()]
        grads = torch.autograd.grad(call(x), [x, *params], create_graph=True)
        return torch.autograd.grad(sum(g.to(x.dtype).float().square().sum() if x.dtype != torch.float64 else g.square().sum()
                                       for g in grads), [x, *params], allow_unused=True)

    def fused(x):
        normed, rest = PA.layer_norm_residual(x, ln)
        y, n = PA.mlp_residual(normed, rest, layers, after if next_norm else None)
        assert (n is not None) == next_norm
        return (y * dy).sum() + ((n * dn).sum() if next_norm else 0)

    mods64 = [copy.deepcopy(m).double() for m in modules]

    def plain(x):
        y = x + mods64[1](mods64[0](x))
        return (y * dy.double()).sum() + ((mods64[2](y) * dn.double()).sum() if next_norm else 0)

    want = second(mods64, x.double(), plain)
    names = ["x"] + [f"{k}.{n}" for k, m in enumerate(modules) for n, _ in m.named_parameters()]
    for dtype in (torch.float32, torch.bfloat16):
        for m in modules:
            m.to(dtype)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == torch.float32):
            got = second(modules, x, fused)
        for name, g, w in zip(names, got, want):
            if w is None or w.norm() == 0:  # a sum that does not depend on the last bias
                assert g is None or g.float().norm() <= 1e-6 * want[1].norm()
                continue
            # every chain passes the block four times, with some ten bf16 roundings (1.1e-3 of a value each on the average)
            # of terms that cancel by a few; the parts that used to be missing are of the size of the result
            assert_rel_l2(g, w, name + " " + str(dtype), tol=4e-2)
    out = fused(x.detach().requires_grad_(True))
    with torch.no_grad():
        layers[0].bias.add_(1.0)
    params = list(layers.parameters())
    with pytest.raises(RuntimeError, match="modified"):
        torch.autograd.grad(out, params, create_graph=True, retain_graph=True)


@pytest.mark.parametrize("C,S,B,N,grid", [(256, 64, 2, 1001, None), (128, 16, 1, 33, None), (256, 32, 1, 12 * 9, (12, 9))])
def test_bf16_blocks_with_fused_tails_train_like_separate_ones(C, S, B, N, grid):
    """A chain of two bf16 blocks and its head: residuals and LayerNorms in the layer's and the MLP's kernels are no
    further from the float32 model than the same blocks with a hook on their layers, which makes the layer a call of its own."""
    announce("fused training tails", C, S, B, N, grid)
    torch.manual_seed(N)
    kw = dict(functional_dim=3, embedding_dim=2, out_dim=3, n_layers=2, n_hidden=C, n_head=C // 32, mlp_ratio=2, slice_num=S,
              structured_shape=grid, use_te=False)
    model = pn.Transolver(**kw).cuda().train()
    x, e = torch.randn(B, N, 3, device="cuda"), torch.rand(B, N, 2, device="cuda")
    dy = torch.randn(B, N, 3, device="cuda")

    def step(amp=True):
        model.zero_grad(set_to_none=True)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=amp):
            out = model(x, e)
        (out.float() * dy).sum().backward()
        return out.detach().float(), {n: p.grad.clone() for n, p in model.named_parameters()}

    out, got = step()
    seen = []
    handles = [b.Attn.register_forward_hook(lambda *a: seen.append(1)) for b in model.blocks]
    apart_out, apart = step()
    for h in handles:
        h.remove()
    assert len(seen) == 2
    want_out, want = step(amp=False)
    # both are bf16 chains of the same length; the fused one rounds no more often, so its error differs by chance only:
    # over the thousands of elements of each of these vectors by a few per cent (a gradient of four elements alone, the
    # temperature's at 33 points, can be off by any factor)
    flat = lambda grads: torch.cat([grads[n].reshape(-1) for n in want]).cpu()
    for got_v, apart_v, want_v in ((out, apart_out, want_out), (flat(got), flat(apart), flat(want))):
        e_got, e_apart = to.rel_l2(got_v.cpu(), want_v.cpu()), to.rel_l2(apart_v.cpu(), want_v.cpu())
        assert e_got <= 1.3 * e_apart, (e_got, e_apart)


@pytest.mark.parametrize("C,S,B,grid", [(256, 64, 2, (21, 17)), (256, 64, 3, (64, 96)), (128, 16, 1, (3, 11)), (256, 32, 1, (8, 4)),
                                        (128, 128, 2, (9, 30)), (256, 128, 1, (16, 20))])
def test_structured_training_forward_with_and_without_the_block_tail(C, S, B, grid):
    """The hand-back on float32 tokens with the residual and LayerNorm in the same call, at full and ragged tiles, several
    batch elements, more tiles than workgroups, and at 128 slices, where it runs as separate kernels: against the same
    layer followed by the residual add and LayerNorm in float64."""
    announce("structured training forward", C, S, B, grid)
    torch.manual_seed(S)
    N, H = grid[0] * grid[1], C // 32
    ref, hip = make_pair("structured2d", C, H, 32, S, spatial=grid, sharpen=3.0)
    hip.train()
    ln = torch.nn.LayerNorm(C).cuda()
    with torch.no_grad():
        ln.weight.add_(0.3 * torch.randn(C, device="cuda")), ln.bias.add_(0.3 * torch.randn(C, device="cuda"))
        for m in (ref, hip):
            m.out_linear.weight.copy_(m.out_linear.weight.bfloat16().float())
    x, res = torch.randn(2, B, N, C, device="cuda").bfloat16()
    y = hip(x).detach()
    fx, normed = (t.detach() for t in hip.forward_block_with_grad(x, res, ln))
    want = y.double() + res.double()
    # the tail adds the residual to a result rounded once (2^-9 / sqrt(3) = 1.1e-3), or not at all, and rounds the sum
    assert_rel_l2(fx, want, "y + residual", tol=3e-3)
    assert_rel_l2(normed, torch.nn.functional.layer_norm(fx.double(), (C,), ln.weight.double(), ln.bias.double()), "LayerNorm",
                  tol=3e-3)
    if C * N <= 100_000:
        assert_rel_l2(y, ref(x.float().cpu()), "y", tol=1e-2)


def test_output_dropout_in_training_matches_the_reference_site():
    """The reference applies nn.Dropout to the layer output in training mode (physics_attention.py:499): kept entries
    are y / (1 - p), the rest zero, gradients flow through the kept entries only; eval mode is the identity."""
    announce("output dropout in training")
    torch.manual_seed(0)
    layer = pn.PhysicsAttentionIrregularMesh(64, heads=2, dim_head=32, dropout=0.25, slice_num=16, use_te=False).cuda()
    x = torch.randn(2, 2000, 64, device="cuda")
    layer.eval()
    with torch.no_grad():
        y_eval = layer(x)
    layer.train()
    xg = x.clone().requires_grad_(True)
    y = layer(xg)
    kept = y != 0
    frac = kept.float().mean().item()
    assert abs(frac - 0.75) < 0.01, frac
    assert_fp32_close(y[kept], (y_eval / 0.75)[kept], "kept entries")
    y.sum().backward()
    assert xg.grad is not None and torch.isfinite(xg.grad).all()
    blk = pn.TransolverBlock(2, 64, 0.25, mlp_ratio=2, slice_num=16, use_te=False).cuda().train()
    out = blk(x)
    assert out.shape == x.shape and torch.isfinite(out).all()


def test_modules_with_hooks_are_called_in_training():
    """Hooks on a block's MLP, its Linears and the output head run in a float32 training step (weight and spectral
    normalisation form the weight in one), and the gradients are those of the step without hooks."""
    announce("hooks in float32 training")
    torch.manual_seed(0)
    model = pn.Transolver(functional_dim=3, embedding_dim=2, out_dim=3, n_layers=2, n_hidden=64, n_head=4, mlp_ratio=2,
                          slice_num=32, use_te=False).cuda().train()
    x, e, dy = (torch.randn(2, 300, n, device="cuda") for n in (3, 2, 3))

    def step():
        model.zero_grad(set_to_none=True)
        (model(x, e) * dy).sum().backward()
        return {n: p.grad.clone() for n, p in model.named_parameters()}

    want = step()
    block, mlp = model.blocks[1], model.blocks[1].ln_mlp1[1]
    hooked = [block.ln_mlp2, *block.ln_mlp2, mlp, mlp.layers, *mlp.layers, model.preprocess.layers[0]]
    for m in hooked:
        seen = []
        handle = m.register_forward_hook(lambda *a: seen.append(1))
        got = step()
        handle.remove()
        assert len(seen) == 1, m
        for n in want:  # the same products in float32, in another order
            assert_rel_l2(got[n], want[n].cpu(), n, tol=1e-4)
    torch.nn.utils.parametrizations.weight_norm(mlp.layers[0])
    want_w = mlp.layers[0].weight.detach().clone()
    with torch.no_grad():
        mlp.layers[0].parametrizations.weight.original0.mul_(2.0)
    seen = []
    handle = mlp.layers[0].register_forward_hook(lambda m, i, o: seen.append((i[0].detach(), o.detach(), m.bias.detach())))
    step()
    handle.remove()
    inp, out, bias = seen[0]
    assert_rel_l2(out, (inp @ (2.0 * want_w).t() + bias).cpu(), "normalised weight", tol=1e-5)


def test_head_of_a_bf16_block_is_called_where_it_is_more_than_a_layernorm_and_a_linear():
    """The last block by itself and in its model, bf16 training: hooks on ln_mlp2 and its modules run, a first module of
    another kind is called."""
    announce("hooks on the head of a bf16 block")
    torch.manual_seed(0)
    model = pn.Transolver(functional_dim=3, embedding_dim=2, out_dim=3, n_layers=1, n_hidden=256, n_head=8, mlp_ratio=2,
                          slice_num=32, use_te=False).cuda().train()
    block = model.blocks[0]
    x, e = torch.randn(2, 300, 3, device="cuda"), torch.rand(2, 300, 2, device="cuda")
    rows = 2 * torch.randn(2, 300, 256, device="cuda").bfloat16()
    runs = (lambda: block(rows.clone().requires_grad_(True)), lambda: model(x, e))
    with torch.autocast("cuda", dtype=torch.bfloat16):
        for run in runs:
            want = run()
            for m in (block.ln_mlp2, *block.ln_mlp2):
                seen = []
                handle = m.register_forward_hook(lambda *a: seen.append(1))
                got = run()
                handle.remove()
                assert len(seen) == 1, m
                assert_rel_l2(got, want, "output with a hook", tol=1e-2)  # a LayerNorm from rounded rows, or unrounded ones
        block.ln_mlp2[0] = torch.nn.Identity()
        for run in runs:
            seen = []
            handle = block.ln_mlp2[1].register_forward_hook(lambda m, i, o: seen.append((i[0].float(), o.float())))
            out = run()
            handle.remove()
            assert torch.equal(seen[0][1], out.float())
            std = seen[0][0].std().item()
            assert not 0.9 < std < 1.1, std  # rows that nothing normalised


def test_mlp_module_differentiates_twice_and_forward():
    """An Mlp by itself, float32: gradients of gradients, forward mode, torch.func, and the refusal of another type."""
    announce("second derivatives of the Mlp")
    torch.manual_seed(0)
    net = Mlp(4, 64, 8).cuda()
    ref = copy.deepcopy(net).cpu().double()
    x = torch.randn(5000, 4, device="cuda")

    def second(m, x):
        x = x.detach().requires_grad_(True)
        (gx,) = torch.autograd.grad(m(x).square().sum(), x, create_graph=True)
        return torch.autograd.grad(gx.square().sum(), [x, *m.parameters()])

    for got, want in zip(second(net, x), second(ref, x.cpu().double())):
        # float32 sums over 5 000 rows: 5000^0.5 * 2^-24 = 4e-6 of the terms, which cancel by up to ten
        assert_rel_l2(got, want.float(), "second derivative", tol=4e-5)
    t = torch.randn_like(x)
    _, jvp = torch.func.jvp(net, (x,), (t,))
    _, want = torch.func.jvp(ref, (x.cpu().double(),), (t.cpu().double(),))
    assert_rel_l2(jvp.detach(), want.detach().float(), "jvp", tol=1e-5)
    got = torch.func.vmap(torch.func.grad(lambda v: net(v).sum()))(x[:8])
    want = torch.func.vmap(torch.func.grad(lambda v: ref(v).sum()))(x[:8].cpu().double())
    assert_rel_l2(got, want.float(), "vmap of grad", tol=1e-5)
    with pytest.raises(RuntimeError):
        net(x.bfloat16())


@pytest.mark.parametrize("variant", ["irregular", "plus", "structured2d", "block"])
def test_parameters_may_change_between_the_passes(variant):
    """The gradients of a bf16 training step are those of the parameters its forward saw, whatever is done to the parameters
    before the backward."""
    announce("parameters changed between the passes", variant)
    torch.manual_seed(0)
    kw = dict(heads=4, dim_head=32, slice_num=32, use_te=False)
    if variant == "block":
        layer = pn.TransolverBlock(8, 256, 0.0, mlp_ratio=2, slice_num=32, use_te=False)
    elif variant == "structured2d":
        layer = pn.PhysicsAttentionStructuredMesh2D(128, (9, 15), kernel=3, **kw)
    else:
        layer = pn.PhysicsAttentionIrregularMesh(128, plus=variant == "plus", **kw)
    layer = layer.cuda().train()
    C = 256 if variant == "block" else 128
    x, dy = torch.randn(2, 2, 135, C, device="cuda").bfloat16()
    noise = torch.rand(2, 135, 4, 32, device="cuda").bfloat16()
    # the LayerNorms' own weights are saved tensors, as in torch
    params = [p for n, p in layer.named_parameters() if n.split(".")[0] not in ("ln_1",) and not n.startswith("ln_mlp1.0")]

    def step(change):
        xi = x.clone().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer.forward_with_noise(xi, noise) if variant == "plus" else layer(xi)
        if change:
            with torch.no_grad():
                for p in params:
                    p.add_(1.0)
        grads = torch.autograd.grad(y, [xi, *params], dy)
        if change:
            with torch.no_grad():
                for p in params:
                    p.sub_(1.0)
        return grads

    for a, b in zip(step(False), step(True)):
        assert torch.equal(a, b)


def test_mlp_module_under_autocast_leaves_types_that_autocast_leaves():
    """A float64 Mlp in training under bf16 autocast computes in float64, whole numbers are refused."""
    announce("Mlp types under autocast")
    torch.manual_seed(0)
    net, x = Mlp(4, 64, 8).cuda().double(), torch.randn(500, 4, device="cuda", dtype=torch.float64)
    want = net.layers(x)
    with torch.autocast("cuda", dtype=torch.bfloat16):
        got = net(x)
        assert got.dtype == torch.float64 and torch.equal(got, want)
        with pytest.raises(RuntimeError):
            net.float()(torch.ones(5, 4, device="cuda", dtype=torch.int64))


@pytest.mark.parametrize("plus", [False, True])
def test_bf16_training_of_a_layer_left_on_the_host(plus):
    """Parameters in host memory are copied to the input's device in the forward; their gradients cannot be delivered there
    and the backward says so.  Uniform samples of another shape are refused."""
    announce("layer left on the host", plus)
    torch.manual_seed(0)
    layer = pn.PhysicsAttentionIrregularMesh(128, heads=4, dim_head=32, slice_num=32, use_te=False, plus=plus).train()
    x, noise = torch.randn(2, 131, 128, device="cuda").bfloat16(), torch.rand(2, 131, 4, 32, device="cuda").bfloat16()
    run = lambda m: m.forward_with_noise(x, noise) if plus else m(x)
    y = run(layer)
    with pytest.raises(RuntimeError, match="device"):
        y.backward(torch.ones_like(y))
    assert torch.equal(run(copy.deepcopy(layer).cuda()), y)
    if plus:
        with pytest.raises(ValueError, match="uniform"):
            layer.cuda().forward_with_noise(x, noise[:, :100])


@pytest.mark.parametrize("plus", [False, True])
def test_bf16_training_takes_parameters_and_gradients_off_16_byte_boundaries(plus):
    """Parameters that are views into one flat vector, an input and an output gradient that start one element into their
    storage: bit for bit the results of the aligned call."""
    announce("misaligned parameters", plus)
    torch.manual_seed(0)
    layer = pn.PhysicsAttentionIrregularMesh(128, heads=4, dim_head=32, slice_num=32, use_te=False, plus=plus).cuda().train()
    x, dy = torch.randn(2, 2, 131, 128, device="cuda").bfloat16()
    noise = torch.rand(2, 131, 4, 32, device="cuda").bfloat16()

    def off(t):
        flat = torch.empty(t.numel() + 1, dtype=t.dtype, device=t.device)
        flat[1:] = t.detach().reshape(-1)
        return flat[1:].view(t.shape)

    def step(move):
        xi = move(x).detach().requires_grad_(True)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            y = layer.forward_with_noise(xi, move(noise)) if plus else layer(xi)
        return [y.detach()] + list(torch.autograd.grad(y, [xi, *layer.parameters()], move(dy), allow_unused=True))

    want = step(lambda t: t)
    for p in layer.parameters():
        p.data = off(p.data)
    for a, b in zip(step(off), want):
        assert (a is None) == (b is None) and (a is None or torch.equal(a, b))


@pytest.mark.parametrize("rows,c_out,bias", [(4096, 256, True), (4127, 256, False), (16387, 512, True), (33001, 256, True)])
def test_row_gemm_of_256_inputs_with_two_workgroups_per_cu(rows, c_out, bias):
    """The natural-output row GEMM at its smallest row count, ragged last tiles, fewer and more tiles than workgroups."""
    announce("row GEMM, 256 inputs", rows, c_out, bias)
    torch.manual_seed(rows)
    x, w = torch.randn(1, rows, 256, device="cuda").bfloat16(), torch.randn(c_out, 256, device="cuda").bfloat16()
    b = torch.randn(c_out, device="cuda") if bias else None
    y = PF.rows_gemm(x, w, b, PF.LayerDims(1, rows, 256, 8, 32, 64), 256, c_out)
    want = x[0].double().cpu() @ w.double().cpu().t() + (b.double().cpu() if bias else 0)
    # float32 sums, rounded to bf16 once: at most half a unit in the last place (2^-9) of a value, sums far below it
    err = (y[0].double().cpu() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 1e-3).all()


@pytest.mark.parametrize("rows,c_out,bias", [(4096, 256, True), (8193, 256, False), (12320, 512, True), (41007, 256, True)])
def test_row_gemm_of_512_inputs_through_the_ring(rows, c_out, bias):
    """Half the workgroups of a round, a second round of one row, more tiles per workgroup than the ring has stages (both widths)."""
    announce("row GEMM, 512 inputs", rows, c_out, bias)
    torch.manual_seed(rows)
    x, w = torch.randn(1, rows, 512, device="cuda").bfloat16(), torch.randn(c_out, 512, device="cuda").bfloat16()
    b = torch.randn(c_out, device="cuda") if bias else None
    y = PF.rows_gemm(x, w, b, PF.LayerDims(1, rows, 512, 16, 32, 64), 512, c_out)
    want = x[0].double().cpu() @ w.double().cpu().t() + (b.double().cpu() if bias else 0)
    # as above: one rounding to bf16
    err = (y[0].double().cpu() - want).abs()
    assert (err <= 2.0 ** -8 * want.abs() + 1e-3).all()


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("rows,c_in,c_out,bias", [(1, 1, 1, True), (63, 3, 5, False), (65, 5, 66, True), (130, 17, 64, True), (200, 33, 30, True)])
def test_row_gemm_of_odd_inputs(dtype, rows, c_in, c_out, bias):
    """Rows that are no whole 16-byte units: last rows, inputs and outputs of tiles of 64 x 16 x 64, one block of inputs and more."""
    announce("row GEMM, odd inputs", dtype, rows, c_in, c_out, bias)
    torch.manual_seed(rows)
    x, w = torch.randn(1, rows, c_in, device="cuda").to(dtype), torch.randn(c_out, c_in, device="cuda").to(dtype)
    b = torch.randn(c_out, device="cuda") if bias else None
    y = PF.rows_gemm(x, w, b, PF.LayerDims(1, rows, c_in, 1, 1, 1), c_in, c_out)
    want = x[0].double().cpu() @ w.double().cpu().t() + (b.double().cpu() if bias else 0)
    # float32 sums of at most 34 terms of a few units each; bf16 results are rounded once
    err = (y[0].double().cpu() - want).abs()
    assert (err <= (2.0 ** -8 if dtype == torch.bfloat16 else 2.0 ** -22) * want.abs() + 1e-4).all()


@pytest.mark.parametrize("rows,Fh", [(1, 64), (300, 192), (2500, 1024), (14450, 1024), (32768, 1024), (40000, 1024), (70000, 512)])
def test_hidden_gradients_do_not_depend_on_how_the_hidden_units_are_split(rows, Fh):
    """Rows choose how many parts the hidden units are taken in; each row's values have the same bits as in a call of few rows."""
    announce("hidden gradients by split", rows, Fh)
    C, dev = 256, torch.device("cuda")
    gen = torch.Generator().manual_seed(rows)
    rnd = lambda *n: torch.randn(*n, generator=gen)
    u, dy = rnd(rows, C).bfloat16().to(dev), rnd(rows, C).bfloat16().to(dev)
    w1, w2, b1 = (rnd(Fh, C) / 16).bfloat16().to(dev), (rnd(C, Fh) / 16).bfloat16().to(dev), (0.1 * rnd(Fh)).to(dev)
    act, dh = PF.mlp_backward(u, dy, w1, b1, w2)
    for part in (slice(0, min(rows, 200)), slice(max(0, rows - 300), rows)):
        few_act, few_dh = PF.mlp_backward(u[part].contiguous(), dy[part].contiguous(), w1, b1, w2)
        assert torch.equal(act[part], few_act) and torch.equal(dh[part], few_dh)


@pytest.mark.parametrize("rows,Fh", [(1, 256), (63, 1024), (64, 320), (65, 256), (2000, 1024), (32768, 256), (32769, 256), (65537, 64),
                                     (2 * 256 * 128 + 1, 256)])
def test_norm_mlp_backward_against_float64(rows, Fh):
    """d x of y = x + Mlp(LayerNorm(x)) with the product that ends in the LayerNorm's backward in one kernel: blocks of 64 rows up
    to 32 768 rows (256 compute units), of 128 beyond, workgroups with one block and with several, ragged last blocks."""
    announce("norm mlp backward", rows, Fh)
    C, eps, dev = 256, 1e-5, torch.device("cuda")
    assert PF.norm_mlp_backward_supported(torch.bfloat16, rows, C, Fh)
    gen = torch.Generator().manual_seed(rows + Fh)
    rnd = lambda *n: torch.randn(*n, generator=gen)
    x, dy = (2 * rnd(rows, C) + 0.5).bfloat16().to(dev), rnd(rows, C).bfloat16().to(dev)
    w1, w2 = (rnd(Fh, C) / C ** 0.5).bfloat16().to(dev), (rnd(C, Fh) / Fh ** 0.5).bfloat16().to(dev)
    b1, gam, bet = (0.1 * rnd(Fh)).to(dev), (0.5 + torch.rand(C, generator=gen)).to(dev), (0.1 * rnd(C)).to(dev)
    u = F.layer_norm(x.float(), (C,), gam, bet, eps).bfloat16()
    dx, d_w1, d_b1, d_w2, d_b2, d_g, d_b = PF.norm_mlp_backward(u, dy, x, w1, b1, w2, gam, eps)
    # the same formulas in float64 from the same bf16 inputs (u as the kernel's producer rounded it)
    xd, ud, dyd = x.double(), u.double(), dy.double()
    h = ud @ w1.double().t() + b1.double()
    phi = 0.5 * (1 + torch.erf(h / 2 ** 0.5))
    dh = (dyd @ w2.double()) * (phi + h * torch.exp(-h * h / 2) / (2 * torch.pi) ** 0.5)
    dn = dh @ w1.double()
    centred = xd - xd.mean(-1, keepdim=True)
    rstd = torch.rsqrt(centred.square().mean(-1, keepdim=True) + eps)
    xh, gg = centred * rstd, dn * gam.double()
    want = rstd * (gg - gg.mean(-1, keepdim=True) - xh * (gg * xh).mean(-1, keepdim=True)) + dyd
    # dx is rounded once (1.7e-3), dh, gelu(h) and dn before it; sums over rows average those roundings out, but for few rows
    assert_rel_l2(dx, want, "d x", 4e-3)
    assert_rel_l2(d_w1, dh.t() @ ud, "d w1", 4e-3)
    assert_rel_l2(d_b1, dh.sum(0), "d b1", 4e-3)
    assert_rel_l2(d_w2, dyd.t() @ (h * phi), "d w2", 4e-3)
    assert_rel_l2(d_b2, dyd.sum(0), "d b2", 1e-5)
    assert_rel_l2(d_g, (dn * xh).sum(0), "d gamma", 6e-3)
    assert_rel_l2(d_b, dn.sum(0), "d beta", 6e-3)


def test_norm_mlp_backward_of_few_rows_with_infinities_keeps_them_where_they_are():
    """A row with an infinite gradient leaves the other rows' d x as they are; rows past the end add nothing."""
    C, Fh, rows, dev = 256, 256, 70, torch.device("cuda")
    torch.manual_seed(0)
    x, dy = torch.randn(rows, C, device=dev).bfloat16(), torch.randn(rows, C, device=dev).bfloat16()
    w1, w2 = (torch.randn(Fh, C, device=dev) / 16).bfloat16(), (torch.randn(C, Fh, device=dev) / 16).bfloat16()
    b1, gam = torch.zeros(Fh, device=dev), torch.ones(C, device=dev)
    u = F.layer_norm(x.float(), (C,)).bfloat16()
    clean = PF.norm_mlp_backward(u, dy, x, w1, b1, w2, gam, 0.0)
    dy[rows - 1, 3] = float("inf")
    dirty = PF.norm_mlp_backward(u, dy, x, w1, b1, w2, gam, 0.0)
    assert all(torch.isfinite(t.float()).all() for t in clean)
    assert torch.equal(clean[0][:rows - 1], dirty[0][:rows - 1]) and not torch.isfinite(dirty[0][rows - 1].float()).all()


@pytest.mark.parametrize("kind,dim,heads,dim_head,S,grid,kernel,N", [
    ("irregular", 64, 2, 16, 32, None, 0, 1), ("irregular", 36, 3, 20, 8, None, 0, 333), ("irregular", 128, 8, 16, 64, None, 0, 2500),
    ("structured2d", 128, 8, 16, 32, (13, 11), 3, 143), ("structured2d", 32, 4, 8, 16, (9, 14), 5, 126),
    ("structured3d", 64, 4, 16, 32, (5, 6, 7), 3, 210),
])
def test_fp32_layer_in_two_calls_against_the_stages(monkeypatch, kind, dim, heads, dim_head, S, grid, kernel, N):
    """A float32 layer's training step in one library call each way against the same stages called one by one: widths off the
    tiles of 32 that turn the weights around, every tap, few and many partial sums, temperatures at and beyond the clamp."""
    announce("fp32 train calls", kind, dim, heads, dim_head, S, grid)
    temps = [0.2 + 5.6 * i / (heads - 1) for i in range(heads)]
    temps[-1] = 5.0
    kw = {} if grid is None else dict(spatial=grid, kernel=kernel)
    _, hip = make_pair(kind, dim, heads, dim_head, S, sharpen=2.0, temps=temps, **kw)
    hip.train()
    x0, dy = torch.randn(2, N, dim, device="cuda"), torch.randn(2, N, dim, device="cuda")

    def step():
        x = x0.clone().requires_grad_(True)
        hip.zero_grad(set_to_none=True)
        y = hip(x)
        y.backward(dy)
        return [y.detach(), x.grad] + [p.grad.clone() for p in hip.parameters()]

    assert PF.layer_train_supported(torch.float32, hip.layer_dims(x0))
    got = step()
    monkeypatch.setattr(PF, "layer_train_supported", lambda *a, **k: False)
    want = step()
    for g, w in zip(got, want):
        assert_rel_l2(g, w, "two calls against the stages", 2e-6)



@pytest.mark.parametrize("B,N,C,S", [(1, 1, 256, 64), (3, 33, 256, 64), (1, 8229, 256, 32), (17, 40, 256, 16), (130, 33, 256, 64),
                                     (1, 32_761, 128, 64), (513, 33, 128, 16), (5, 6571, 128, 32), (2, 4127, 256, 16)])
def test_point_stage_with_its_products_against_the_stages(B, N, C, S):
    """The irregular layer's backward, whose per-point kernel forms the projections and d out_x itself, against the stages with
    these in memory: single points, ragged tiles, few and many batch elements, workgroups without a tile, every S.  Both
    round the three products to bf16 from float32 sums in different orders; where the rounding falls the other way (2^-8 of a
    value, one in ten at most) the results differ by 2^-8 sqrt(0.1) = 1.2e-3, the sums with cancelling terms by more."""
    announce("point stage with products", B, N, C, S)
    from physicsnemo_amd import autograd as PA
    torch.manual_seed(S + N)
    H = C // 32
    _, hip = make_pair("irregular", C, H, 32, S, temps=[0.3 + 0.4 * k for k in range(H)])
    x, dy = torch.randn(2, B, N, C, device="cuda").bfloat16()
    dims, kp = hip.layer_dims(x), hip.kernel_params(torch.bfloat16, x.device)
    names = dict(hip.named_parameters())
    params = [names[n.replace("_weight", ".weight").replace("_bias", ".bias")] for n in PA._LAYER_PARAMS]
    xc = x.clone().requires_grad_(True)
    PA.PhysicsAttentionMfmaFunction.apply(xc, dims, None, *params).backward(dy)

    st = PF.MfmaStages(kp, dims, x.device)
    st.pack_params()
    st.project_softmax(x)
    st.slice_reduce()
    st.combine_attention()
    linear = PF.LayerDims(B, N, C, H, 32, S)
    x_mid, fx_mid = PF.project_inputs(x, kp, dims)
    g = PF.rows_gemm(dy, kp["out_linear_weight"].view(C, C).t().contiguous(), None, linear, C, C)
    d_tok, _, _ = PF.output_backward(st.w_pack, dy, st.tok_out, kp["out_linear_weight"], dims)
    d_num, d_norm, _ = PF.slice_attention_backward(st.tok, st.norm, d_tok, kp, dims)
    d_proj, d_ws, d_bs, d_temp = PF.point_backward(x_mid, fx_mid, g, st.tok_out, d_num, d_norm, kp, dims)
    w_t = torch.cat([kp["in_project_x_weight"].view(C, C).t(), kp["in_project_fx_weight"].view(C, C).t()], dim=1).contiguous()
    assert_rel_l2(xc.grad, PF.rows_gemm(d_proj, w_t, None, linear, 2 * C, C), "dx", tol=4e-3)
    rows, d_b = d_proj.float().reshape(-1, 2 * C), d_proj.double().reshape(-1, 2 * C).sum(0)
    d_w = rows.t() @ x.float().reshape(-1, C)
    assert_rel_l2(hip.in_project_x.weight.grad, d_w[:C], "d W_x", tol=4e-3)
    assert_rel_l2(hip.in_project_fx.weight.grad, d_w[C:], "d W_fx", tol=4e-3)
    assert_rel_l2(hip.in_project_fx.bias.grad, d_b[C:], "d b_fx", tol=4e-3)
    assert_rel_l2(hip.in_project_slice.weight.grad, d_ws.view(S, 32), "d W_slice", tol=4e-3)
    assert_rel_l2(hip.in_project_slice.bias.grad, d_bs, "d b_slice", tol=2e-2)
    assert_rel_l2(hip.temperature.grad.reshape(-1), d_temp.reshape(-1), "d temperature", tol=2e-2)


@pytest.mark.parametrize("linear1,linear2,through_norm", [(False, False, True), (True, False, True), (False, True, False)])
def test_frozen_parts_of_a_norm_mlp_are_not_differentiated(monkeypatch, linear1, linear2, through_norm):
    """Gradients of frozen Linears (and, with LayerNorm and input frozen too, the way through it) are not formed: the call hands
    back None for them and leaves their memory alone, a block's backward asks for what its parameters need, and what is formed
    has the same bits."""
    announce("frozen norm mlp", linear1, linear2, through_norm)
    torch.manual_seed(3)
    C, Fh, rows = 256, 512, 3000
    ln = torch.nn.LayerNorm(C).cuda()
    layers = torch.nn.Sequential(torch.nn.Linear(C, Fh), torch.nn.GELU(), torch.nn.Linear(Fh, C)).cuda()
    x, dy = torch.randn(2, rows, C, device="cuda").bfloat16()
    asked, call = [], PF.norm_mlp_backward

    def spy(*args, **kw):
        asked.append((args, call(*args, **kw)))
        return asked[-1][1]

    monkeypatch.setattr(PF, "norm_mlp_backward", spy)

    def step(frozen):
        for part, on in ((layers[0], linear1), (layers[2], linear2), (ln, through_norm)):
            part.requires_grad_(on or not frozen)
        for p in [*ln.parameters(), *layers.parameters()]:
            p.grad = None
        xi = x.clone().requires_grad_(through_norm or not frozen)
        with torch.autocast("cuda", dtype=torch.bfloat16):
            normed = torch.nn.functional.layer_norm(x.float(), (C,), ln.weight, ln.bias, ln.eps).detach().bfloat16()
            assert PA.norm_mlp_fused(xi, ln, layers)
            y, _ = PA.norm_mlp_residual_of(xi, normed, ln, layers)
        y.backward(dy)
        return [xi.grad] + [p.grad for p in [*layers.parameters(), *ln.parameters()]]

    every = step(False)
    part = step(True)
    _, formed = asked[-1]
    on = [through_norm, linear1, linear1, linear2, linear2, through_norm, through_norm]
    assert [t is not None for t in formed] == on
    for a, b, wanted in zip(every, part, on):
        assert (b is None) if not wanted else torch.equal(a, b)


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
def test_parameters_may_be_freed_between_the_passes(dtype):
    """Sharded training frees a layer's parameters between its passes: the gradients have the shapes that the parameters had in
    the forward pass."""
    announce("parameters freed between the passes", dtype)
    torch.manual_seed(0)
    hip = pn.PhysicsAttentionIrregularMesh(128, heads=4, dim_head=32, slice_num=32, use_te=False).cuda()
    x, dy = torch.randn(2, 1, 300, 128, device="cuda").to(dtype)
    params = list(hip.parameters())

    def grads(change):
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == torch.bfloat16):
            y = hip(x)
        kept = [p.data for p in params]
        change()
        out = torch.autograd.grad(y, params, dy)
        for p, k in zip(params, kept):
            p.data = k
        return out

    def free():
        for p in params:
            p.data = torch.empty(0, device="cuda")

    for g, w, p in zip(grads(free), grads(lambda: None), params):
        assert g.shape == p.shape and g.dtype == torch.float32 and torch.equal(g, w)


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
def test_blocks_in_training_call_what_is_watched_or_replaced(dtype):
    """A hook on a layer's dropout or on every module, a replaced forward of the dropout or of the layer: a training block calls
    them, once per pass, and the result is that of the block without them."""
    announce("watched dropouts", dtype)
    torch.manual_seed(0)
    C = 128
    block = pn.TransolverBlock(4, C, 0.0, mlp_ratio=1, slice_num=32, use_te=False).cuda()
    attn, drop, seen = block.Attn, block.Attn.out_dropout, []
    x = torch.randn(2, 700, C, device="cuda").to(dtype).requires_grad_(True)

    def step():
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == torch.bfloat16):
            return block(x)

    def watch(m, *_):
        if m is attn or m is drop:
            seen.append(m)

    def replaced(m):
        plain = type(m).forward
        m.forward = lambda t: (seen.append(m), plain(m, t))[1]
        return lambda: m.__dict__.pop("forward")

    want = step()
    everywhere = torch.nn.modules.module.register_module_forward_hook
    for start, whom in ((lambda: drop.register_forward_hook(watch).remove, [drop]),
                        (lambda: everywhere(watch).remove, [drop, attn]),
                        (lambda: replaced(drop), [drop]), (lambda: replaced(attn), [attn])):
        seen.clear()
        end = start()
        try:
            got = step()
        finally:
            end()
        assert seen == whom
        assert_rel_l2(got, want, "block", tol=1e-6 if dtype == torch.float32 else 5e-3)  # bf16: LayerNorm from rounded rows
        got.float().sum().backward()


def test_training_call_refuses_parameters_of_another_type():
    """The library reads the parameters by the type that goes with the activations: 16-bit ones for float32 activations (half the
    memory it would read), a 16-bit bias, weights of two types are errors."""
    announce("training call, parameter types")
    hip = pn.PhysicsAttentionIrregularMesh(64, heads=2, dim_head=32, slice_num=32, use_te=False).cuda()
    x = torch.randn(1, 100, 64, device="cuda")
    dims, names = hip.layer_dims(x), dict(hip.named_parameters())
    params = {n: names[n.replace("_weight", ".weight").replace("_bias", ".bias")].detach() for n in PA._LAYER_PARAMS}
    assert torch.isfinite(PF.layer_train_forward(x, None, params, dims)[0]).all()
    halves = {n: p.bfloat16() if n in PA._LARGE else p for n, p in params.items()}
    for wrong in (halves, {**params, "out_linear_bias": params["out_linear_bias"].bfloat16()},
                  {**params, "in_project_x_weight": params["in_project_x_weight"].bfloat16()}):
        with pytest.raises(TypeError):
            PF.layer_train_forward(x, None, wrong, dims)


@pytest.mark.parametrize("next_norm", [False, True])
def test_norm_mlp_block_differentiates_twice(next_norm):
    """x + Mlp(LayerNorm(x)) in one function, as model blocks of 256 channels train, LayerNorm(x) given without a graph: gradients
    of a function of its gradient, by x and every parameter of the LayerNorm before, the Linears and the LayerNorm behind,
    against float64.  A parameter of any of them that changed between the passes is refused there and only there."""
    announce("norm mlp twice", next_norm)
    torch.manual_seed(1)
    rows, C, Fh = 300, 256, 128
    ln, after = torch.nn.LayerNorm(C, eps=1e-3).cuda(), torch.nn.LayerNorm(C).cuda()
    layers = torch.nn.Sequential(torch.nn.Linear(C, Fh), torch.nn.GELU(), torch.nn.Linear(Fh, C)).cuda()
    modules = [ln, layers] + ([after] if next_norm else [])
    with torch.no_grad():
        for m in modules:
            for p in m.parameters():
                p.copy_((p + 0.1 * torch.randn_like(p)).bfloat16().float())
    x, dy, dn = (torch.randn(rows, C, device="cuda").bfloat16() for _ in range(3))

    def second(mods, x, call):
        x = x.detach().requires_grad_(True)
        params = [p for m in mods for p in m.parameters()]
        grads = torch.autograd.grad(call(x), [x, *params], create_graph=True)
        return torch.autograd.grad(sum(g.to(x.dtype).float().square().sum() if x.dtype != torch.float64 else g.square().sum()
                                       for g in grads), [x, *params], allow_unused=True)

    def fused(x):
        assert PA.norm_mlp_fused(x, ln, layers)
        normed = F.layer_norm(x.detach().float(), (C,), ln.weight.detach().float(), ln.bias.detach().float(), ln.eps).bfloat16()
        y, n = PA.norm_mlp_residual_of(x, normed, ln, layers, after if next_norm else None)
        assert (n is not None) == next_norm
        return (y * dy).sum() + ((n * dn).sum() if next_norm else 0)

    mods64 = [copy.deepcopy(m).double() for m in modules]

    def plain(x):
        y = x + mods64[1](mods64[0](x))
        return (y * dy.double()).sum() + ((mods64[2](y) * dn.double()).sum() if next_norm else 0)

    want = second(mods64, x.double(), plain)
    names = ["x"] + [f"{k}.{n}" for k, m in enumerate(modules) for n, _ in m.named_parameters()]
    for dtype in (torch.float32, torch.bfloat16):
        for m in modules:
            m.to(dtype)
        with torch.autocast("cuda", dtype=torch.bfloat16, enabled=dtype == torch.float32):
            got = second(modules, x, fused)
        for name, g, w in zip(names, got, want):
            if w is None or w.norm() == 0:  # a sum that does not depend on the last bias
                assert g is None or g.float().norm() <= 1e-6 * want[1].norm()
                continue
            # four passes through the block with some ten bf16 roundings each (1.1e-3 of a value) of terms that cancel by a few
            assert_rel_l2(g, w, name + " " + str(dtype), tol=4e-2)
    for m in modules:  # float32 parameters: what the plain backward reads of them are copies in bf16
        m.float()
    every = [x.detach().requires_grad_(True), *(p for m in modules for p in m.parameters())]
    for changed in (ln.weight, ln.bias, layers[0].weight, layers[0].bias, layers[2].weight, *([after.weight] if next_norm else [])):
        with torch.autocast("cuda", dtype=torch.bfloat16):
            out = fused(every[0])
        first = torch.autograd.grad(out, every, retain_graph=True)
        with torch.no_grad():
            changed.add_(0.5)
        if changed is not after.weight:
            for g, w in zip(torch.autograd.grad(out, every, retain_graph=True), first):
                assert torch.equal(g, w)
        with pytest.raises(RuntimeError, match="modified"):
            torch.autograd.grad(out, every, create_graph=True)


def _oracle64_gradients(hip, kind, dim, heads, dim_head, S, x, dy, spatial=None, kernel=3):
    """x's gradient and the parameters' by autograd over the float64 oracle with the layer's parameters."""
    if kind == "irregular":
        ref = to.OraclePhysicsAttentionIrregularMesh(dim, heads=heads, dim_head=dim_head, slice_num=S)
    else:
        cls = to.OraclePhysicsAttentionStructuredMesh2D if kind == "structured2d" else to.OraclePhysicsAttentionStructuredMesh3D
        ref = cls(dim, spatial, heads=heads, dim_head=dim_head, slice_num=S, kernel=kernel)
    ref = ref.to(x.device).double()
    ref.load_state_dict({k: v.double() for k, v in hip.state_dict().items()})
    xd = x.detach().double().requires_grad_(True)
    ref(xd).backward(dy.double())
    return {"x": xd.grad, **{n: p.grad for n, p in ref.named_parameters()}}


@pytest.mark.parametrize("B,N,C,S", [(2, 3001, 256, 64), (1, 9000, 256, 32), (3, 700, 256, 16), (1, 33_000, 128, 64), (2, 17_000, 128, 16)])
def test_point_stage_with_its_products_is_as_close_to_float64_as_the_stages(B, N, C, S):
    """The irregular layer's gradients in bf16 against float64: the kernel that forms x_mid, fx_mid and d out_x itself rounds to
    bf16 what the stages with these in memory round, so that its errors are theirs but for single roundings that fall the other
    way (one in a few thousand values, whose float32 sums differ in their last bits): less than 2 % apart over four seeds."""
    announce("point stage with products against float64", B, N, C, S)
    H = C // 32
    names = ["x", "in_project_x.weight", "in_project_x.bias", "in_project_fx.weight", "in_project_fx.bias", "in_project_slice.weight",
             "in_project_slice.bias", "temperature"]
    square = {n: [0.0, 0.0] for n in names}
    for seed in range(4):
        _, hip = make_pair("irregular", C, H, 32, S, seed=seed, temps=[0.3 + 0.4 * k for k in range(H)])
        hip.train()
        x, dy = torch.randn(2, B, N, C, device="cuda").bfloat16()
        want = _oracle64_gradients(hip, "irregular", C, H, 32, S, x, dy)
        xr = x.clone().requires_grad_(True)
        hip.zero_grad(set_to_none=True)
        hip(xr).backward(dy)
        one = {"x": xr.grad, **{n: p.grad for n, p in hip.named_parameters()}}

        dims, kp = hip.layer_dims(x), hip.kernel_params(torch.bfloat16, x.device)
        st = PF.MfmaStages(kp, dims, x.device)
        st.pack_params()
        st.project_softmax(x)
        st.slice_reduce()
        st.combine_attention()
        linear = PF.LayerDims(B, N, C, H, 32, S)
        x_mid, fx_mid = PF.project_inputs(x, kp, dims)
        g = PF.rows_gemm(dy, kp["out_linear_weight"].view(C, C).t().contiguous(), None, linear, C, C)
        d_tok, _, _ = PF.output_backward(st.w_pack, dy, st.tok_out, kp["out_linear_weight"], dims)
        d_num, d_norm, _ = PF.slice_attention_backward(st.tok, st.norm, d_tok, kp, dims)
        d_proj, d_ws, d_bs, d_t = PF.point_backward(x_mid, fx_mid, g, st.tok_out, d_num, d_norm, kp, dims)
        w_t = torch.cat([kp["in_project_x_weight"].view(C, C).t(), kp["in_project_fx_weight"].view(C, C).t()], dim=1).contiguous()
        d_w, d_b = PF.cols_gemm(d_proj, x, col_sums=True)
        apart = [PF.rows_gemm(d_proj, w_t, None, linear, 2 * C, C), d_w[:C], d_b[:C], d_w[C:], d_b[C:], d_ws, d_bs, d_t]
        for n, a in zip(names, apart):
            w = want[n].reshape(-1)
            for k, got in enumerate((one[n], a)):
                square[n][k] += ((got.double().reshape(-1) - w).norm() / w.norm()).item() ** 2
    for n, (one, apart) in square.items():
        assert one <= 1.02 ** 2 * apart, (n, (one / 4) ** 0.5, (apart / 4) ** 0.5)


@pytest.mark.parametrize("kind,dim,heads,dim_head,S,grid,kernel,N", [
    ("irregular", 64, 2, 16, 32, None, 0, 1), ("irregular", 36, 3, 20, 8, None, 0, 333), ("irregular", 128, 8, 16, 64, None, 0, 2500),
    ("structured2d", 128, 8, 16, 32, (13, 11), 3, 143), ("structured2d", 32, 4, 8, 16, (9, 14), 5, 126),
    ("structured3d", 64, 4, 16, 32, (5, 6, 7), 3, 210),
])
def test_fp32_layer_in_two_calls_against_float64(kind, dim, heads, dim_head, S, grid, kernel, N):
    """Every gradient of a float32 layer's training step against float64: up to 1.5e-6 was seen for these shapes, 4.1e-6 for d
    temperature, whose terms cancel most; four times that."""
    announce("fp32 train calls against float64", kind, dim, heads, dim_head, S, grid)
    temps = [0.2 + 5.6 * i / (heads - 1) for i in range(heads)]
    kw = {} if grid is None else dict(spatial=grid, kernel=kernel)
    _, hip = make_pair(kind, dim, heads, dim_head, S, sharpen=2.0, temps=temps, **kw)
    hip.train()
    x, dy = torch.randn(2, 2, N, dim, device="cuda")
    assert PF.layer_train_supported(torch.float32, hip.layer_dims(x))
    want = _oracle64_gradients(hip, kind, dim, heads, dim_head, S, x, dy, **kw)
    xr = x.clone().requires_grad_(True)
    hip(xr).backward(dy)
    for n, got in [("x", xr.grad)] + [(n, p.grad) for n, p in hip.named_parameters()]:
        err = (got.double() - want[n]).norm() / want[n].norm().clamp(min=1e-30)
        assert err <= (1.7e-5 if n == "temperature" else 6e-6), (n, err.item())


@pytest.mark.parametrize("dim,heads,N", [(48, 3, 17), (128, 8, 15), (128, 8, 16), (256, 16, 33), (32, 2, 9000), (128, 8, 9000)])
def test_fp32_layer_of_16_channel_heads_at_the_edges_of_its_tiles(dim, heads, N):
    """The per-point kernels of 16-channel heads and 32 slices (tiles of 16 points): the same bounds."""
    test_fp32_layer_in_two_calls_against_float64("irregular", dim, heads, 16, 32, None, 0, N)


@pytest.mark.parametrize("dtype,C,O", [(torch.float32, 128, 132), (torch.float32, 64, 256), (torch.bfloat16, 128, 256)])
@pytest.mark.parametrize("grid,B", [((1, 1), 70), ((2, 3), 11), ((1, 31), 2), ((32, 1), 3), ((2, 2, 2), 9), ((3, 4, 5), 7)])
def test_conv_weight_gradient_of_grids_within_a_block_of_rows(dtype, C, O, grid, B):
    """Grids of fewer points than the 32 rows that a step advances by: several batch elements within one step."""
    announce("conv weight gradient, tiny grids", dtype, C, O, grid, B)
    torch.manual_seed(B)
    N, k = int(np.prod(grid)), 3
    g, x = torch.randn(B, N, O, device="cuda").to(dtype), torch.randn(B, N, C, device="cuda").to(dtype)
    dims = PF.LayerDims(B, N, C, 4, 32, 32, grid[0], grid[1], k, grid[2] if len(grid) == 3 else 0, 1)
    dw, db = PF.cols_gemm(g, x, col_sums=True, grid=dims)
    w = torch.zeros(O, C, *(k,) * len(grid), dtype=torch.float64, requires_grad=True)
    conv = torch.nn.functional.conv2d if len(grid) == 2 else torch.nn.functional.conv3d
    conv(x.double().cpu().transpose(1, 2).reshape(B, C, *grid), w, padding=1).backward(
        g.double().cpu().transpose(1, 2).reshape(B, O, *grid))
    assert_fp32_close(dw, w.grad, "d weight")
    assert_fp32_close(db, g.double().sum((0, 1)), "d bias")


@pytest.mark.parametrize("rows,ca,cb", [(1, 128, 128), (33, 132, 64), (2015, 256, 128), (4129, 64, 260)])
def test_float32_weight_gradient_with_infinities_at_the_ends_of_chunks(rows, ca, cb):
    """What lies behind a chunk of rows, the next chunk's or nothing, reads as zero: an infinity in the last row stays in its
    column and one in the first row does too."""
    announce("float32 infinities", rows, ca, cb)
    a, b = (1 + torch.rand(rows, c, device="cuda") for c in (ca, cb))
    for row in (0, rows - 1):
        for inf_in_a in (False, True):
            x, y = a.clone(), b.clone()
            (x if inf_in_a else y)[row, 5] = float("inf")
            got, sums = PF.cols_gemm(x, y, col_sums=True)
            want = torch.zeros(ca, cb, dtype=torch.bool, device="cuda")
            (want[5] if inf_in_a else want[:, 5]).fill_(True)
            assert not got.isnan().any() and torch.equal(got.isinf(), want)
            assert not sums.isnan().any() and sums.isinf().sum() == int(inf_in_a)


@pytest.mark.parametrize("grid,C,O,B", [((110, 140), 32, 256, 1), ((60, 57), 64, 128, 10), ((101, 63), 96, 128, 2)])
def test_float32_convolution_in_tall_and_flat_tiles(grid, C, O, B):
    """Row counts on either side of the rule between 128 and 64 rows a workgroup, one to three steps per tap: against float64, to
    the rounding of the sums (as above)."""
    announce("float32 conv tiles", grid, C, O, B)
    torch.manual_seed(C)
    N = int(np.prod(grid))
    dims = PF.LayerDims(B, N, C, O // 32, 32, 32, grid[0], grid[1], 3, 0, 1)
    x, w = torch.randn(B, N, C, device="cuda"), torch.randn(O, C, 3, 3, device="cuda") / (9 * C) ** 0.5
    got = PF.rows_gemm(x, w.movedim(1, -1).contiguous(), None, dims, C, O)
    want = torch.nn.functional.conv2d(x.double().transpose(1, 2).reshape(B, C, *grid).cpu(), w.double().cpu(), padding=1)
    assert_rel_l2(got, want.reshape(B, O, N).transpose(1, 2), "conv", tol=4e-6)


@pytest.mark.parametrize("off", [-float("inf"), torch.finfo(torch.float32).min, -1e38])
@pytest.mark.parametrize("dim,heads,dim_head,S,N", [(128, 8, 16, 32, 333), (48, 3, 16, 32, 17), (64, 4, 16, 64, 333), (96, 3, 32, 32, 65)])
def test_fp32_training_with_a_slice_switched_off(dim, heads, dim_head, S, N, off):
    """A slice of no weight adds nothing to any gradient: outputs and gradients are those of float64 with a finite bias that leaves it
    no weight either (of -inf itself, autograd's d temperature is 0 inf = NaN).  The bounds are those of the layers without one."""
    announce("fp32 training, a slice off", dim, heads, dim_head, S, N, off)
    ref, hip = make_pair("irregular", dim, heads, dim_head, S, sharpen=2.0, temps=[0.2 + 5.6 * i / (heads - 1) for i in range(heads)])
    hip.train()
    x, dy = torch.randn(2, 2, N, dim, device="cuda")
    with torch.no_grad():
        hip.in_project_slice.bias[5] = -1e30
    want = _oracle64_gradients(hip, "irregular", dim, heads, dim_head, S, x, dy)
    ref.load_state_dict({k: v.cpu() for k, v in hip.state_dict().items()})
    with torch.no_grad():
        want_y = ref.double()(x.double().cpu())
        hip.in_project_slice.bias[5] = off
    xr = x.clone().requires_grad_(True)
    y = hip(xr)
    y.backward(dy)
    assert ((y.double().cpu() - want_y).norm() / want_y.norm()).item() <= 6e-6
    for n, got in [("x", xr.grad)] + [(n, p.grad) for n, p in hip.named_parameters()]:
        err = (got.double() - want[n]).norm() / want[n].norm().clamp(min=1e-30)
        assert err <= (1.7e-5 if n == "temperature" else 6e-6), (n, err.item())
