"""RMSNorm / LayerNorm rows and the column sums of the training composites against fp64: widths of one to the most
vectors per lane and with idle lanes, tokens around the waves of a launch, with and without parameters, joined gradient;
and the composites (feed-forward block, SwiGLU block, the gated attention between norm and output) against the same
layers with one parameter frozen, which runs them operator by operator."""
import numpy as np
import pytest
import torch
import torch.nn.functional as F

import fairseq_apollo_amd as M
from gpu_util import DEV

pytestmark = pytest.mark.gpu
# one rounding of the result (2^-9 bf16, 2^-11 fp16) on values up to a few times the rms; fp32: sums of up to 8200 terms
# in fp32, sqrt(8200) 2^-24 of the sum of magnitudes at worst
ULP = {torch.bfloat16: 2 ** -8, torch.float16: 2 ** -10, torch.float32: 4e-6}


def _close(got, ref, dtype, scale=None):
    ref = ref.double().cpu()
    scale = ref.abs() + ref.pow(2).mean().sqrt() if scale is None else scale.double().cpu()
    assert got.dtype == dtype and got.shape == ref.shape
    assert bool(((got.double().cpu() - ref).abs() <= ULP[dtype] * scale + 1e-12).all())


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,D,affine", [(1, 8, True), (5, 520, True), (2100, 1024, True), (67, 2048, True), (8200, 256, False)])
@pytest.mark.parametrize("kind", [M.ops.TOKEN_RMSNORM, M.ops.TOKEN_LAYERNORM])
def test_row_norm_both_ways(dtype, T, D, affine, kind):
    torch.manual_seed(T + D)
    x, dy, add = (torch.randn(T, D, device=DEV).to(dtype) + (0.5 if i == 0 else 0) for i in range(3))
    w = (torch.randn(D, device=DEV) * 0.3).to(dtype) if affine else None
    b = torch.randn(D, device=DEV).to(dtype) if affine and kind == M.ops.TOKEN_LAYERNORM else None
    leaves = [t.double().cpu().requires_grad_(True) if t is not None else None for t in (x, w, b)]
    x64, w64, b64 = leaves
    c64 = x64 - x64.mean(-1, keepdim=True) if kind == M.ops.TOKEN_LAYERNORM else x64
    y64 = c64 * torch.rsqrt(c64.pow(2).mean(-1, keepdim=True) + 1e-5)
    y64 = y64 if w64 is None else y64 * (w64 + 1)
    y64 = y64 if b64 is None else y64 + b64
    y64.backward(dy.double().cpu())
    args = [t.clone().requires_grad_(True) if t is not None else None for t in (x, w, b)]
    assert M.modules.row_norm_covers(*args)
    y = M.modules.row_norm(args[0], kind, args[1], args[2], 1e-5)
    _close(y, y64.detach(), dtype)
    y.backward(dy)
    _close(args[0].grad, x64.grad, dtype)
    with torch.no_grad():
        hat = ((c64 * torch.rsqrt(c64.pow(2).mean(-1, keepdim=True) + 1e-5)).detach().abs() * dy.double().cpu().abs()).sum(0)
    if w is not None:
        _close(args[1].grad, w64.grad, dtype, hat + w64.grad.abs())
    if b is not None:
        _close(args[2].grad, b64.grad, dtype, dy.double().cpu().abs().sum(0))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("D,ffn,T,norm", [(64, 96, 33, 'layernorm'), (256, 520, 700, 'rmsnorm')])
def test_feed_forward_composite(dtype, D, ffn, T, norm):
    """Against fp64 of the same formula."""
    torch.manual_seed(D)
    block = M.NormalizedFeedForwardNetwork(D, ffn, norm_type=norm).to(DEV).to(dtype).train()
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0, 0.1)
    x = torch.randn(2, T, D, device=DEV).to(dtype).requires_grad_(True)
    dy = torch.randn(2, T, D, device=DEV).to(dtype)
    assert block._one_operator(x)
    y = block(x)
    y.backward(dy)
    P = {k: v.detach().double().cpu().requires_grad_(True) for k, v in block.named_parameters()}
    x64 = x.detach().double().cpu().requires_grad_(True)
    n = M.modules.row_norm_formula(x64, M.ops.TOKEN_LAYERNORM, P['norm.weight'], P['norm.bias'], 1e-5) if norm == 'layernorm' \
        else x64 * torch.rsqrt(x64.pow(2).mean(-1, keepdim=True) + 1e-5) * (P['norm.weight'] + 1)
    y64 = x64 + F.silu(n @ P['fc1.weight'].t() + P['fc1.bias']) @ P['fc2.weight'].t()
    y64.backward(dy.double().cpu())
    # four roundings in a row on the way to any result: 4 ulp of the rms and of the value
    for got, ref in [(y, y64), (x.grad, x64.grad)] + [(p.grad, P[k].grad) for k, p in block.named_parameters()]:
        _close(got.detach(), ref.detach(), dtype, 4 * (ref.detach().abs() + ref.detach().pow(2).mean().sqrt()))


@pytest.mark.parametrize("dtype,D,S,E,heads,L,chunk,act,two", [
    (torch.bfloat16, 64, 32, 128, 1, 96, 32, 'rmsnorm', False), (torch.float16, 128, 64, 64, 2, 130, -1, 'silu', False),
    (torch.float32, 64, 16, 96, 1, 70, -1, 'rmsnorm', True)])
def test_mix_composite_matches_the_operators(dtype, D, S, E, heads, L, chunk, act, two):
    """The composite against the operators one by one (taken when a parameter is frozen): the same values in other
    kernels, roundings apart."""
    torch.manual_seed(S)
    layer = M.MovingAverageGatedAttention(D, S, E, 8, chunk_size=chunk, moving_act=act, norm_num_groups=4, num_heads=heads,
                                          bidirectional=two).to(DEV).to(dtype).train()
    with torch.no_grad():
        for p in layer.parameters():
            if not bool(p.any()):
                p.normal_(0, 0.2)
    x0, dy = (torch.randn(2, L, D, device=DEV).to(dtype) for _ in range(2))
    mask = torch.arange(L, device=DEV)[None, :] >= torch.tensor([[L], [L - 9]], device=DEV) if two else None
    out = []
    for freeze in (False, True):
        layer.h_proj.weight.requires_grad_(not freeze)
        layer.zero_grad()
        x = x0.clone().requires_grad_(True)
        y, _ = layer(x, mask)
        assert ("MixOut" in type(y.grad_fn).__name__) == (not freeze)
        y.backward(dy if mask is None else dy * (~mask)[..., None])
        out.append([y.detach(), x.grad] + [p.grad for n, p in layer.named_parameters() if n != 'h_proj.weight'])
    for a, b in zip(*out):
        # the same formulas in both: a handful of roundings of intermediate results apart, 8 ulp of the rms and of the value
        b64 = b.double().cpu()
        _close(a, b64, dtype, 8 * (b64.abs() + b64.pow(2).mean().sqrt()))


@pytest.mark.parametrize("norm", [M.layers.RMSNorm, M.layers.LayerNorm])
def test_norms_under_transforms(norm):
    """Function transforms, forward-mode tangents and tracing see torch's own operations: the values of the same module
    on the CPU, fp32 sums of 64 terms in another order apart (sqrt(64) 2^-24 of the sum of magnitudes)."""
    torch.manual_seed(3)
    cpu = norm(64)
    with torch.no_grad():
        for p in cpu.parameters():
            p.normal_(0, 0.3)
    dev = norm(64).to(DEV)
    dev.load_state_dict(cpu.state_dict())
    x, t = torch.randn(4, 7, 64), torch.randn(4, 7, 64)
    xd, td = x.to(DEV), t.to(DEV)

    def near(got, ref):
        _close(got.detach(), ref.detach(), torch.float32)

    near(torch.func.vmap(dev)(xd), cpu(x))
    want = torch.func.jvp(cpu, (x,), (t,))
    for a, b in zip(torch.func.jvp(dev, (xd,), (td,)), want):
        near(a, b)
    near(torch.func.grad(lambda v: (dev(v) * td).sum())(xd), torch.func.grad(lambda v: (cpu(v) * t).sum())(x))
    with torch.autograd.forward_ad.dual_level():
        dual = dev(torch.autograd.forward_ad.make_dual(xd, td))
        near(torch.autograd.forward_ad.unpack_dual(dual).tangent, want[1])
    traced = torch.jit.trace(dev, xd, check_trace=False)
    near(traced(td), cpu(t))


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("first,second", [(True, True), (False, False), (False, True)])
def test_feed_forward_of_other_projections(dtype, first, second):
    """Projections with and without a bias where the constructor builds the other form: every bias enters the result and
    gets its gradient.  Against fp64 of the same formula.  These run operator by operator: eight results in a row are
    rounded on the longest way (weight + 1, norm, product, activation and back through the product, the activation, the
    norm and the sum with the residual's share): 8 ulp of the rms and of the value."""
    D, ffn, T = 64, 96, 33
    torch.manual_seed(2)
    block = M.NormalizedFeedForwardNetwork(D, ffn)
    block.fc1, block.fc2 = torch.nn.Linear(D, ffn, bias=first), torch.nn.Linear(ffn, D, bias=second)
    block = block.to(DEV).to(dtype).train()
    with torch.no_grad():
        for p in block.parameters():
            p.normal_(0, 0.1)
    x = torch.randn(2, T, D, device=DEV).to(dtype).requires_grad_(True)
    dy = torch.randn(2, T, D, device=DEV).to(dtype)
    y = block(x)
    y.backward(dy)
    P = {k: v.detach().double().cpu().requires_grad_(True) for k, v in block.named_parameters()}
    x64 = x.detach().double().cpu().requires_grad_(True)
    n = F.layer_norm(x64, (D,), P['norm.weight'] + 1, P['norm.bias'], 1e-5)
    y64 = x64 + F.linear(F.silu(F.linear(n, P['fc1.weight'], P.get('fc1.bias'))), P['fc2.weight'], P.get('fc2.bias'))
    y64.backward(dy.double().cpu())
    for got, ref in [(y, y64), (x.grad, x64.grad)] + [(p.grad, P[k].grad) for k, p in block.named_parameters()]:
        _close(got.detach(), ref.detach(), dtype, 8 * (ref.detach().abs() + ref.detach().pow(2).mean().sqrt()))


@pytest.mark.parametrize("name,bias", [("h_proj", True), ("v_proj", False), ("mx_proj", False)])
def test_gated_attention_of_other_projections(name, bias):
    """The gated attention with a projection of the other form against the operators one by one (a frozen parameter) in
    fp32; sums of up to 300 terms in another order: 8 ulp of the rms and of the value, as in the test above."""
    torch.manual_seed(4)
    layer = M.MovingAverageGatedAttention(64, 32, 128, 8, chunk_size=32, norm_num_groups=4)
    old = getattr(layer, name)
    setattr(layer, name, torch.nn.Linear(old.in_features, old.out_features, bias=bias))
    layer = layer.to(DEV).train()
    with torch.no_grad():
        for p in layer.parameters():
            if not bool(p.any()):
                p.normal_(0, 0.2)
    x0, dy = (torch.randn(2, 96, 64, device=DEV) for _ in range(2))
    out = []
    for freeze in (False, True):
        layer.gamma.requires_grad_(not freeze)
        layer.zero_grad()
        x = x0.clone().requires_grad_(True)
        y, _ = layer(x)
        y.backward(dy)
        out.append([y.detach(), x.grad] + [p.grad for n, p in layer.named_parameters() if n != 'gamma'])
    for a, b in zip(*out):
        assert a is not None and b is not None
        b64 = b.double().cpu()
        _close(a, b64, torch.float32, 8 * (b64.abs() + b64.pow(2).mean().sqrt()))
    if bias:                                               # the result without the bias is another one
        with torch.no_grad():
            layer.h_proj.bias.zero_()
        assert not torch.allclose(layer(x0)[0], out[0][0], rtol=1e-3, atol=1e-3)


@pytest.mark.parametrize("change", ["forward", "global"])
def test_composites_of_replaced_forwards(change):
    """Modules whose `forward` was replaced on the instance, and hooks on every module of the program, are called in
    training wherever the operators one by one call them (fc1, v_proj and mx_proj run there as products of their own)."""
    torch.manual_seed(4)
    layer = M.Mega2Layer(64, 32, 128, 8, 96, 32, norm_num_groups=4, moving_act='rmsnorm').to(DEV).train()
    block = M.NormalizedFeedForwardNetwork(64, 96).to(DEV).train()
    seen = [layer.attn.move_act, layer.attn.h_proj, layer.ffn.w1, layer.ffn.w3, block.norm]
    x, calls = torch.randn(2, 96, 64, device=DEV), []
    want = [layer(x).detach(), block(x).detach()]
    if change == "forward":
        for m in seen:
            m.forward = lambda v, m=m, f=m.forward: calls.append(m) or f(v)
        got = [layer(x), block(x)]
    else:
        handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: calls.append(m))
        try:
            got = [layer(x), block(x)]
        finally:
            handle.remove()
    assert all(sum(c is m for c in calls) == 1 for m in seen)
    for a, b in zip(got, want):
        b64 = b.double().cpu()
        _close(a.detach(), b64, torch.float32, 8 * (b64.abs() + b64.pow(2).mean().sqrt()))


def _through_cat(y):
    """y on the way to a concatenation behind one element: its gradient is a contiguous view that starts on no 16 bytes."""
    return torch.cat([torch.zeros(1, dtype=y.dtype, device=y.device), y.flatten()])


@pytest.mark.parametrize("what", ["layernorm", "rmsnorm", "feed-forward", "swiglu", "gated attention"])
def test_gradients_off_16_bytes(what):
    """The same gradients whether the incoming one starts on 16 bytes or not."""
    torch.manual_seed(9)
    module = {"layernorm": lambda: M.layers.LayerNorm(64), "rmsnorm": lambda: M.layers.RMSNorm(64),
              "feed-forward": lambda: M.NormalizedFeedForwardNetwork(64, 96), "swiglu": lambda: M.SwiGLU(64, 96),
              "gated attention": lambda: M.MovingAverageGatedAttention(64, 32, 128, 8, chunk_size=32, norm_num_groups=4)}[what]()
    module = module.to(DEV).train()
    x0 = torch.randn(2, 96, 64, device=DEV)
    weight = torch.randn(2 * 96 * 64 + 1, device=DEV)
    out = []
    for off in (True, False):
        module.zero_grad()
        x = x0.clone().requires_grad_(True)
        y = module(x)
        y = y[0] if isinstance(y, tuple) else y
        ((_through_cat(y) * weight).sum() if off else (y * weight[1:].view(y.shape)).sum()).backward()
        out.append([x.grad] + [p.grad for p in module.parameters()])
    for a, b in zip(*out):
        assert torch.equal(a, b)


def test_gated_attention_under_anomaly_detection():
    """Every gradient that leaves a backward pass is written whole: with fresh memory filled with NaN, anomaly detection
    finds none."""
    torch.manual_seed(4)
    layer = M.MovingAverageGatedAttention(64, 32, 128, 8, chunk_size=32, norm_num_groups=4).to(DEV).train()
    x = torch.randn(2, 96, 64, device=DEV, requires_grad=True)
    filled = torch.utils.deterministic.fill_uninitialized_memory
    torch.use_deterministic_algorithms(True, warn_only=True)           # new tensors start as NaN
    torch.utils.deterministic.fill_uninitialized_memory = True
    try:
        with torch.autograd.set_detect_anomaly(True):
            y, _ = layer(x)
            assert "MixOut" in type(y.grad_fn).__name__
            y.square().sum().backward()
    finally:
        torch.use_deterministic_algorithms(False)
        torch.utils.deterministic.fill_uninitialized_memory = filled
    assert all(bool(t.grad.isfinite().all()) for t in (x, *layer.parameters()))


def _second_derivatives(call, formula, tensors):
    """Gradients of sum((d loss / d inputs)^2) by both: `call` on the GPU in fp32, `formula` on the CPU in fp64."""
    out = []
    for f, t in ((call, [v.clone().requires_grad_(True) for v in tensors]),
                 (formula, [v.double().cpu().requires_grad_(True) for v in tensors])):
        y = f(*t)
        y = y if isinstance(y, tuple) else (y,)
        weights = [torch.linspace(-1, 1, v.numel(), dtype=v.dtype).view(v.shape).to(v.device) for v in y]
        first = torch.autograd.grad(y, t, weights, create_graph=True)
        second = torch.autograd.grad(sum(g.square().sum() for g in first), t, materialize_grads=True)
        out.append((first, second))
    for got, ref in zip(out[0][0] + out[0][1], out[1][0] + out[1][1]):
        ref = ref.detach()
        # sums of up to 66 x 100 products in fp32, twice in a row
        _close(got.detach(), ref, torch.float32, 16 * (ref.abs() + ref.pow(2).mean().sqrt()))


@pytest.mark.parametrize("kind", [M.ops.TOKEN_RMSNORM, M.ops.TOKEN_LAYERNORM])
def test_second_derivatives_feed_forward(kind):
    torch.manual_seed(6)
    x, nw, w1, b1, w2 = (torch.randn(*s, device=DEV) * 0.5 for s in ((2, 33, 64), (64,), (96, 64), (96,), (64, 96)))
    nb = torch.randn(64, device=DEV) if kind == M.ops.TOKEN_LAYERNORM else None
    tensors = [x, nw, w1 * 0.2, b1, w2 * 0.2] + ([nb] if nb is not None else [])

    def formula(x, nw, w1, b1, w2, nb=None):
        c = x - x.mean(-1, keepdim=True) if nb is not None else x
        n = c * torch.rsqrt(c.pow(2).mean(-1, keepdim=True) + 1e-5) * (nw + 1)
        return x + F.linear(F.silu(F.linear(n if nb is None else n + nb, w1, b1)), w2)

    _second_derivatives(lambda x, nw, w1, b1, w2, nb=None: M.modules.FeedForwardFunc.apply(x, nw, nb, w1, b1, w2, kind, 1e-5),
                        formula, tensors)


@pytest.mark.parametrize("residual", [False, True])
def test_second_derivatives_swiglu(residual):
    torch.manual_seed(7)
    x, res, w1, w3, w2 = (torch.randn(*s, device=DEV) * 0.3 for s in ((2, 33, 64), (2, 33, 64), (96, 64), (96, 64), (64, 96)))

    def formula(x, w1, w3, w2, res=None):
        y = F.linear(F.silu(F.linear(x, w1)) * F.linear(x, w3), w2)
        return y if res is None else y + res

    _second_derivatives(lambda x, w1, w3, w2, res=None: M.modules.SwiGLUBlockFunc.apply(x, res, w1, w3, w2), formula,
                        [x, w1, w3, w2] + ([res] if residual else []))


@pytest.mark.parametrize("act,heads", [(M.ops.TOKEN_RMSNORM, 1), (M.ops.TOKEN_SILU, 2)])
def test_second_derivatives_gated_attention(act, heads):
    """The two halves of the gated attention around the attention itself (here: the sum of q, k and v columns)."""
    torch.manual_seed(8)
    B, L, C, D, S, E = 2, 12, 6, 32, 16, 24
    W = 2 * D + S + E
    shapes = ((B, L, D), (B, D, L), (E, D), (E,), (W, D), (W,), (2, S), (2, S), (B, L, D), (D, E))
    tensors = [torch.randn(*s, device=DEV) * 0.3 for s in shapes]
    if act == M.ops.TOKEN_RMSNORM:
        tensors.append(torch.randn(D, device=DEV) * 0.3)
    freqs = torch.rand(S // heads // 2, device=DEV)

    def call(xn, mx, vw, vb, mw, mb, ga, be, res, hw, aw=None):
        v, base, q, k = M.modules.MixInFunc.apply(xn, mx, vw, vb, mw, mb, ga, be, freqs, aw, act, 1e-5, heads, C)
        attn = v.view(B, L, E) + (q * k).sum(-1).view(B, L, 1)
        return M.modules.MixOutFunc.apply(res, base, attn, hw, S)

    def formula(xn, mx, vw, vb, mw, mb, ga, be, res, hw, aw=None):
        v, m = F.silu(F.linear(xn, vw, vb)), mx.transpose(1, 2)
        m = F.silu(m) if aw is None else m * torch.rsqrt(m.pow(2).mean(-1, keepdim=True) + 1e-5) * (aw + 1)
        u, z, r, hx = F.linear(m, mw, mb).split([D, S, E, D], -1)
        z = F.normalize(z, p=2, dim=-1, eps=1e-5)
        ang = (torch.arange(L, dtype=torch.float64) % C)[:, None] * freqs.double().cpu().repeat(heads)
        turn = torch.polar(torch.ones_like(ang), ang)
        q, k = (torch.view_as_real(torch.view_as_complex((z * (ga[i] + 1) + be[i]).reshape(B, L, -1, 2)) * turn).flatten(-2)
                for i in (0, 1))
        attn = v + (q * k).sum(-1, keepdim=True)
        return res + torch.sigmoid(u) * (F.silu(hx + F.linear(attn * F.silu(r), hw)) - res)

    _second_derivatives(call, formula, tensors)


@pytest.mark.parametrize("what", ["feed-forward", "swiglu", "gated attention"])
def test_gradients_asked_for_one_by_one(what):
    """torch.autograd.grad for one input at a time gives the bits of the whole backward pass, and the products behind the
    gradients that nobody asks for are left out (the next test)."""
    torch.manual_seed(9)
    module = {"feed-forward": lambda: M.NormalizedFeedForwardNetwork(64, 96), "swiglu": lambda: M.SwiGLU(64, 96),
              "gated attention": lambda: M.MovingAverageGatedAttention(64, 32, 128, 8, chunk_size=32, norm_num_groups=4,
                                                                       moving_act='rmsnorm')}[what]().to(DEV).train()
    x = torch.randn(2, 96, 64, device=DEV, requires_grad=True)
    dy = torch.randn(2, 96, 64, device=DEV)
    inputs = [x, *(p for p in module.parameters() if p.requires_grad)]

    def run(wanted):
        y = module(x)
        y = y[0] if isinstance(y, tuple) else y
        return torch.autograd.grad(y, wanted, dy)

    whole = run(inputs)
    for t, g in zip(inputs, whole):
        assert torch.equal(run([t])[0], g)


def test_products_nobody_asks_for():
    """The composites' backward passes with one gradient wanted: the others' weights come back as None."""
    H, S = M._lib.load_host(), M.ops._stream(torch.device(DEV))
    torch.manual_seed(1)
    x, n, pre, h, w1, w2 = (torch.randn(*s, device=DEV) for s in ((6, 8), (6, 8), (6, 16), (6, 16), (16, 8), (8, 16)))
    ffn = [x, x, n, pre, h, M.ops.TOKEN_RMSNORM, None, None, 1e-5, w1, w2, S]
    assert [t is not None for t in H.ffn_backward(*ffn, 1)] == [True, False, False, False, True, False]
    assert [t is not None for t in H.ffn_backward(*ffn, 1 << 5)] == [False] * 5 + [True]
    glu = [x, n, pre, h, pre, w1, w1, w2, S]
    assert [t is not None for t in H.swiglu_backward(*glu, 1)] == [True, False, False, False]
    assert [t is not None for t in H.swiglu_backward(*glu, 1 << 4)] == [False, False, False, True]
