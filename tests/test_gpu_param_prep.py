"""The one-launch parameter work of a training step (mega_train_prepare, mega_ema_param_sums + mega_ema_param_finish)
against the operators it stands in for, which the oracle pins (ema_coeffs_fwd / _bwd, norm_params_fwd / _bwd,
ema_backward): state counts that do and do not divide a wave, batches around the four slices the finish kernel cuts them
into, both element types, one- and two-sided, more rows than channels of the norm and fewer."""
import numpy as np
import pytest
import torch

import fairseq_apollo_amd as M
from gpu_util import DEV

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cls,D,N,two,B,L,dtype", [
    (M.MultiHeadComplexEMA, 8, 16, False, 1, 40, torch.float32), (M.MultiHeadComplexEMA, 24, 5, True, 3, 70, torch.float32),
    (M.MultiHeadEMA, 7, 3, True, 5, 33, torch.float32), (M.MultiHeadEMA, 40, 16, False, 9, 65, torch.float32),
    (M.MultiHeadComplexEMA, 16, 1, False, 4, 20, torch.float32), (M.MultiHeadComplexEMA, 16, 7, False, 2, 50, torch.bfloat16),
])
def test_one_launch_parameters_match_the_operators(cls, D, N, two, B, L, dtype):
    torch.manual_seed(D + N)
    move = cls(D, ndim=N, bidirectional=two).to(DEV).to(dtype)
    stored = [t.detach() for t in move._stored()]
    x = torch.randn(B, D, L, device=DEV)
    dy = torch.randn(B, D, L, device=DEV)
    norm = M.TimestepNorm(2 * D, 2, prior_count=3).to(DEV)
    with torch.no_grad():
        for p in norm.parameters():
            p.normal_(0, 0.5)
    layer, (ng, nb, pm, pv, pc) = M.ops.PreparedEMA.of_parameters(
        stored, move.complex, two, True, x, (norm.weight, norm.bias, norm.prior_mean, norm.prior_logv, norm.prior_count), B)
    p, q, g, om = M.ops.ema_coeffs_fwd(*stored, move.complex)
    for a, b in ((layer.p, p), (layer.q, q), (layer.gamma, g), (layer.omega, om)):
        assert torch.equal(a, b)
    want = M.ops.norm_params_fwd(norm.weight, norm.bias, norm.prior_mean, norm.prior_logv, B)
    for a, b in zip((ng, nb, pm, pv), want):
        assert torch.equal(a, b)
    assert pc.tolist() == [3] * B
    ref = M.ops.PreparedEMA(p, torch.view_as_complex(q) if move.complex else q[..., 0],
                            torch.view_as_complex(g) if move.complex else g[..., 0], om, two)
    assert torch.equal(layer(x)[0], ref(x)[0])                     # the same operand images, the same kernels
    got = M._lib.load_host().ema_param_backward(dy, x, None, layer.q, *stored, move.complex, two, True,
                                                M.ops._stream(x.device))
    _, dp, dq, dg, dom = M.ops.ema_backward(dy, x, ref.p, torch.view_as_complex(q) if move.complex else q[..., 0],
                                            torch.view_as_complex(g) if move.complex else g[..., 0], om, layer=ref)
    if move.complex:
        dq, dg = torch.view_as_real(dq.contiguous()), torch.view_as_real(dg.contiguous())
    want = M.ops.ema_coeffs_bwd(dp, dq, dg, dom, *stored[:3], stored[3], stored[4], move.complex)
    # the same fp32 sums over time, added over the batch in another order (B additions of 2^-24 each) and rounded to the
    # parameters' type (2^-9 for bf16)
    tol = 4e-7 * max(B, 4) + (2 ** -8 if dtype is torch.bfloat16 else 0.0)
    for a, b in zip(got, want):
        assert a.shape == b.shape and a.dtype == b.dtype
        scale = float(b.double().abs().max())
        assert float((a.double() - b.double()).abs().max()) <= tol * max(scale, 1e-30)


@pytest.mark.parametrize("dtype,B,L,H,G,masked", [(torch.bfloat16, 2, 33, 128, 4, False), (torch.float16, 3, 257, 256, 16, True),
                                                  (torch.bfloat16, 1, 1, 64, 8, False)])
def test_norm_backward_adds_a_second_gradient(dtype, B, L, H, G, masked):
    """The one-launch form on two gradients gives bit for bit what it gives on their sum rounded to the type."""
    lib = M._lib.load()
    code = M.ops._DT[dtype]
    assert lib.mega_timestep_norm_bwd_adds(code, B, L, H, G) == 1
    torch.manual_seed(L)
    x, a, b = (torch.randn(B, L, H, device=DEV).to(dtype) for _ in range(3))
    mask = (torch.rand(B, L, device=DEV) < 0.2) if masked else None
    pc, pm, pv = torch.zeros(B, dtype=torch.int64, device=DEV), torch.zeros(B, G, device=DEV), torch.ones(B, G, device=DEV)
    gm = torch.randn(H, device=DEV)
    _, cnt, _, _, _, cm, cr = M.ops.group_timestep_norm_fwd(x, pc, pm, pv, gm, gm, mask, G, 1e-5)
    want = M.ops.group_timestep_norm_bwd(a + b, None, None, x, pm, cnt, None, cm, cr, gm, mask, G)
    got = [torch.empty_like(t) for t in want]
    m8 = None if mask is None else mask.view(torch.uint8)
    nws = lib.mega_timestep_norm_bwd_workspace_bytes(code, B, L, H, G)
    ws = torch.empty(nws, dtype=torch.uint8, device=DEV)
    ptr = M.ops._ptr
    rc = lib.mega_group_timestep_norm_bwd_add(ptr(a), ptr(b), None, None, ptr(x), code, ptr(pm), ptr(cnt), None, ptr(cm),
                                              ptr(cr), ptr(gm), ptr(m8), B, L, H, G, *[ptr(t) for t in got], ptr(ws), nws,
                                              M.ops._stream(x.device))
    assert rc == 0, lib.mega_last_error()
    for u, v in zip(got, want):
        assert torch.equal(u, v)
