"""fp32 products on the matrix cores (mega_gemm_f32) against 64-bit products: every storage order, tile and step
remainders, products split along the reduction, epilogues, batched causal forms, values that are not finite; and the
callers that hand their products over (linear layers outside training, attention)."""
import ctypes as C
import math

import pytest
import torch
import torch.nn.functional as F

import fairseq_apollo_amd as M
from gpu_util import DEV

pytestmark = pytest.mark.gpu


class _Gemm(C.Structure):
    _fields_ = [(n, C.c_void_p) for n in ("a", "b", "c", "bias", "residual", "pre")] + \
        [(n, C.c_int64) for n in ("lda", "ldb", "ldc", "ldr", "sa", "sai", "sb", "sbi", "sc", "sci", "M", "N", "K", "batch", "inner")] + \
        [(n, C.c_int32) for n in ("a_kmajor", "b_kmajor", "causal", "silu")] + [("alpha", C.c_float), ("a_padded", C.c_int32)]


def _tol(K):
    """Roundings of the running sum, six for every 32 reduction indices and of either sign, beside the result's own."""
    return 2.0 ** -24 * (2 + math.sqrt(6 * (K / 32 + 1)))


def _call(a, b, c, ka, kb, bias=None, residual=None, silu=False, p=None, alpha=1.0):
    lib = M._lib.load()
    m, n = c.shape
    k = a.shape[0] if ka else a.shape[1]
    ptr = lambda t: None if t is None else t.data_ptr()
    g = _Gemm(ptr(a), ptr(b), ptr(c), ptr(bias), ptr(residual), ptr(p), a.stride(0), b.stride(0), n,
              residual.stride(0) if residual is not None else 0, 0, 0, 0, 0, 0, 0, m, n, k, 1, 1, ka, kb, 0, silu, alpha)
    wide = a.dtype is torch.float32
    nws = lib.mega_gemm_workspace_bytes(m, n, k, 1) if wide else lib.mega_gemm16_workspace_bytes(m, n, k)
    ws = torch.empty(max(nws, 16), dtype=torch.uint8, device=DEV)
    s = torch.cuda.current_stream().cuda_stream
    rc = lib.mega_gemm_f32(C.byref(g), ws.data_ptr(), nws, s) if wide else \
        lib.mega_gemm16(C.byref(g), 1 if a.dtype is torch.bfloat16 else 2, ws.data_ptr(), nws, s)
    assert rc == 0, lib.mega_last_error()
    torch.cuda.synchronize()


def _gemm(a, b, ka, kb, bias=None, residual=None, silu=False, pre=False, alpha=1.0):
    """a [M, K], b [N, K] as given or (ka / kb) stored transposed"""
    m, n = a.shape[1] if ka else a.shape[0], b.shape[1] if kb else b.shape[0]
    c = torch.full((m, n), float("nan"), device=DEV, dtype=a.dtype)
    p = torch.full_like(c, float("nan")) if pre else None
    _call(a, b, c, ka, kb, bias, residual, silu, p, alpha)
    return (c, p) if pre else c


def _rel(x, r):
    return ((x.double() - r).norm() / r.norm().clamp_min(1e-300)).item()


@pytest.mark.parametrize("ka,kb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,wide", [(1, 1, 1, 0), (3, 5, 7, 0), (64, 64, 32, 0), (68, 60, 36, 0), (65, 63, 33, 1), (132, 260, 100, 4),
                                        (36, 4, 132, 0), (300, 140, 2052, 0), (64, 128, 8000, 0), (4100, 4100, 36, 0), (4096, 4224, 64, 4)])
def test_products_of_every_order_and_remainder(m, n, k, wide, ka, kb):
    """wide: columns beside the operands' own in memory (1: rows off 16 bytes)."""
    print(f"case m={m} n={n} k={k} wide={wide} ka={ka} kb={kb}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m + n + k)
    mk = lambda r, c: torch.randn(r, c + wide, generator=gen, device=DEV)[:, :c] * 3
    a, b = mk(k, m) if ka else mk(m, k), mk(k, n) if kb else mk(n, k)
    r = (a.double().t() if ka else a.double()) @ (b.double() if kb else b.double().t())
    assert _rel(_gemm(a, b, ka, kb), r) < _tol(k)


@pytest.mark.parametrize("m,n,k", [(70, 66, 40), (40, 96, 2048), (129, 7, 65)])
def test_epilogues(m, n, k):
    gen = torch.Generator(DEV).manual_seed(5)
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV)
    a, b, bias, res = mk(m, k), mk(n, k), mk(n), mk(m, n)
    r = 0.5 * (a.double() @ b.double().t()) + bias.double() + res.double()
    c, pre = _gemm(a, b, 0, 0, bias, res, True, True, 0.5)
    assert _rel(pre, r) < _tol(k)
    assert _rel(c, F.silu(r)) < _tol(k) + 2.0 ** -22          # (expf and the division: a few units more)


@pytest.mark.parametrize("L,H1,H2", [(64, 8, 12), (100, 16, 20), (260, 64, 128), (1000, 32, 64)])
def test_attention_products_and_gradients(L, H1, H2):
    """q k^T, w v and the four products behind them, causal and not, two heads, against 64 bits."""
    B, Nh = 2, 2
    gen = torch.Generator(DEV).manual_seed(L)
    mk = lambda h: torch.randn(B, L, Nh, h, generator=gen, device=DEV)
    q, k, v, g = mk(H1), mk(H1), mk(H2), mk(H2)
    for causal in (True, False):
        print(f"case L={L} H1={H1} H2={H2} causal={causal}", flush=True)
        assert M.ops.own_attention_products(L, H1, H2, q, k, v)
        y, w = M.ops.attention_fwd(q, k, v, 0.3, 0.0, causal, need_weights=True)
        t = [x.double().transpose(1, 2).contiguous().requires_grad_() for x in (q, k, v)]
        s = 0.3 * (t[0] @ t[1].transpose(-1, -2))
        if causal:
            s = s.masked_fill(torch.ones(L, L, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
        ref = s.softmax(-1) @ t[2]
        ref.backward(g.double().transpose(1, 2))
        got = M.ops.attention_bwd(g, q, k, v, w, 0.3, causal)
        torch.cuda.synchronize()
        # exp of scores with an absolute error of |s| 2^-23 or so, through two more products
        assert _rel(y.transpose(1, 2), ref) < 4e-6
        for x, r in zip(got, t):
            assert _rel(x.transpose(1, 2), r.grad) < 1e-5


def test_values_that_are_not_finite():
    gen = torch.Generator(DEV).manual_seed(9)
    a, b = torch.randn(200, 300, generator=gen, device=DEV), torch.randn(150, 300, generator=gen, device=DEV)
    a[3, 5], a[7, 9], b[11, 100], a[20, 100], b[12, 7] = float("inf"), float("nan"), 3.4e38, 0.25, float("-inf")
    c, r = _gemm(a, b, 0, 0), (a.double() @ b.double().t()).float()
    assert torch.equal(torch.isnan(c), torch.isnan(r)) and torch.equal(torch.isposinf(c), torch.isposinf(r))
    ok = torch.isfinite(r)
    assert _rel(c[ok], r[ok].double()) < _tol(300)


def test_linear_layers_outside_training():
    """project / linear_residual: bias, silu, a residual consumed in place; hooked and replaced layers keep their own call."""
    x, res = torch.randn(3, 50, 96, device=DEV), torch.randn(3, 50, 72, device=DEV)
    lin, nob = torch.nn.Linear(96, 72).to(DEV), torch.nn.Linear(96, 72, bias=False).to(DEV)
    with torch.no_grad():
        r = F.linear(x.double(), lin.weight.double(), lin.bias.double())
        assert M.modules.own_product(lin, x)
        assert _rel(M.modules.project(lin, x), r) < _tol(96)
        assert _rel(M.modules.project(lin, x, True), F.silu(r)) < _tol(96) + 2.0 ** -22
        want = F.linear(x.double(), nob.weight.double()) + res.double()
        assert _rel(M.modules.linear_residual(nob, x, res), want) < _tol(96)
        out = M.modules.linear_residual(nob, x, res, True)
        assert out.data_ptr() == res.data_ptr() and _rel(out, want) < _tol(96)
        hook = lin.register_forward_hook(lambda m, i, o: o * 0)
        assert not M.modules.own_product(lin, x) and not M.modules.project(lin, x).any()
        hook.remove()
        assert not M.modules.own_product(lin, x.transpose(0, 1)) and not M.modules.own_product(lin, x.half())
    assert not M.modules.own_product(lin, x)


@pytest.mark.parametrize("L", [64, 65, 130, 511, 1003])
def test_padded_attention(L):
    """Two-sided attention with padded keys, one row of it padding throughout, at lengths that are whole pieces and not:
    softmax(q k^T) v and its gradients against 64 bits, padded keys getting none."""
    print(f"case L={L}", flush=True)
    B, Nh, H1, H2 = 3, 2, 16, 24
    gen = torch.Generator(DEV).manual_seed(L)
    q, k, v, g = (torch.randn(B, L, Nh, h, generator=gen, device=DEV) for h in (H1, H1, H2, H2))
    mask = torch.zeros(B, L, dtype=torch.bool, device=DEV)
    mask[0, L - L // 3:] = True
    mask[1] = True
    ins = [t.clone().requires_grad_() for t in (q, k, v)]
    y = M.modules.PaddedAttentionFunc.apply(*ins, mask)
    y.backward(g)
    torch.cuda.synchronize()
    ref = [t.double().transpose(1, 2).contiguous().requires_grad_() for t in (q, k, v)]
    s = ref[0] @ ref[1].transpose(-1, -2)
    s = s.masked_fill((mask & ~mask.all(-1, keepdim=True))[:, None, None, :], float("-inf"))
    out = s.softmax(-1) @ ref[2]
    out.backward(g.double().transpose(1, 2))
    assert _rel(y.transpose(1, 2), out) < 4e-6
    for t, r in zip(ins, ref):
        assert _rel(t.grad.transpose(1, 2), r.grad) < 1e-5
    assert not ins[2].grad[0, mask[0]].any() and not ins[1].grad[0, mask[0]].any()


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ka,kb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k,wide", [(8, 8, 8, 0), (64, 64, 64, 0), (72, 56, 40, 8), (136, 264, 104, 0), (1000, 264, 72, 0),
                                        (40, 96, 2056, 0), (264, 1024, 8192, 0), (2048, 1032, 8200, 8)])
def test_16bit_products(dtype, ka, kb, m, n, k, wide):
    """Tile and step remainders, tiles of 128 (the long reductions), parts along the reduction, both types: one rounding
    of a 64-bit product away (2^-9 / 2^-12 of the largest a value can be from its neighbour, half of that on average)."""
    print(f"case {dtype} m={m} n={n} k={k} wide={wide} ka={ka} kb={kb}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m + n + k)
    mk = lambda r, c: torch.randn(r, c + wide, generator=gen, device=DEV).to(dtype)[:, :c]
    a, b = mk(k, m) if ka else mk(m, k), mk(k, n) if kb else mk(n, k)
    r = (a.double().t() if ka else a.double()) @ (b.double() if kb else b.double().t())
    assert _rel(_gemm(a, b, ka, kb), r) < (2.0 ** -9 if dtype is torch.bfloat16 else 2.0 ** -12) + _tol(k)


@pytest.mark.parametrize("m,n,k", [(72, 64, 40), (40, 96, 2048)])
def test_16bit_epilogues(m, n, k):
    """Bias and residual enter before the one rounding, silu acts on the rounded value."""
    gen = torch.Generator(DEV).manual_seed(6)
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(torch.bfloat16)
    a, b, bias, res = mk(m, k), mk(n, k), mk(n), mk(m, n)
    r = a.double() @ b.double().t() + bias.double() + res.double()
    c, pre = _gemm(a, b, 0, 0, bias, res, True, True)
    assert _rel(pre, r) < 2.0 ** -9 + _tol(k)
    assert _rel(c, F.silu(pre.double())) < 2.0 ** -9 + 2.0 ** -22


def _padded_reference(q, k, v, mask):
    s = q.transpose(1, 2).contiguous() @ k.permute(0, 2, 3, 1).contiguous()
    s = s.masked_fill((mask & ~mask.all(-1, keepdim=True))[:, None, None, :], float("-inf"))
    return (s.softmax(-1) @ v.transpose(1, 2).contiguous()).transpose(1, 2)


def test_padded_attention_differentiates_twice_and_in_part():
    """A graph over the backward pass (create_graph) is the formula's, and gradients of some operands are the same values
    as when all are formed; one row is padding throughout."""
    B, L, Nh, H1, H2 = 2, 66, 2, 8, 12
    gen = torch.Generator(DEV).manual_seed(4)
    mk = lambda h: torch.randn(B, L, Nh, h, generator=gen, device=DEV)
    mask = torch.zeros(B, L, dtype=torch.bool, device=DEV)
    mask[0, 50:], mask[1] = True, True
    ins, g, c = [mk(h).requires_grad_() for h in (H1, H1, H2)], mk(H2), mk(H1)
    full = torch.autograd.grad(M.modules.PaddedAttentionFunc.apply(*ins, mask), ins, g)
    for i in range(3):
        part, = torch.autograd.grad(M.modules.PaddedAttentionFunc.apply(*ins, mask), [ins[i]], g)
        assert torch.equal(part, full[i])

    def second(f, ins, g, c):
        dq, = torch.autograd.grad(f(*ins, mask), [ins[0]], g, create_graph=True)
        return torch.autograd.grad((dq * c).sum(), ins)

    got = second(M.modules.PaddedAttentionFunc.apply, ins, g, c)
    ref = [t.detach().double().requires_grad_() for t in ins]
    want = second(_padded_reference, ref, g.double(), c.double())
    for a, b in zip(got, want):
        assert _rel(a, b) < 1e-5                # (as the first derivatives: fp32 products of a softmax's differences)


@pytest.mark.parametrize("m,n,k,own", [(64, 72, 96, True), (64, 70, 96, True), (64, 72, 94, False), (512, 2048, 4096, False)])
def test_fp32_linear_layers_of_sizes_left_to_the_library(m, n, k, own):
    """Odd widths (no whole 16-byte rows) and sizes that the matrix-core kernel serves slower: the module's own call."""
    lin, x = torch.nn.Linear(k, n).to(DEV), torch.randn(m, k, device=DEV)
    with torch.no_grad():
        y = M._lib.load_host().linear_own(x, lin.weight, lin.bias, None, False, False, torch.cuda.current_stream().cuda_stream)
        assert (y is not None) == own
        out = M.modules.project(lin, x)
        assert torch.equal(out, y if own else lin(x))
        assert _rel(out, F.linear(x.double(), lin.weight.double(), lin.bias.double())) < max(_tol(k), 1e-6 * math.sqrt(k / 1024))


@pytest.mark.parametrize("ka,kb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", [(37, 50, 61), (68, 72, 100), (64, 96, 2056), (4096, 4224, 64)])
def test_values_that_are_not_finite_in_every_form(m, n, k, ka, kb):
    """NaN, infinities of either sign and finite values beyond bf16's largest, in every storage order, in element-wise and
    partial steps, in parts along the reduction and in the wide tile: NaN and infinities where the arithmetic has them, the
    other elements as ever."""
    print(f"case m={m} n={n} k={k} ka={ka} kb={kb}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m)
    a, b = torch.randn(m, k, generator=gen, device=DEV), torch.randn(n, k, generator=gen, device=DEV)
    a[3, 5], a[7, k - 1], a[20, 10], b[11, 2], b[n - 1, 7] = float("inf"), float("nan"), 3.4e38, float("-inf"), -3.4e38
    a[20] *= 0.1
    a[20, 10] = 3.4e38
    b[:, 10] *= 0.1
    c = _gemm(a.t().contiguous() if ka else a, b.t().contiguous() if kb else b, ka, kb)
    r = (a.double() @ b.double().t()).float()
    assert torch.equal(torch.isnan(c), torch.isnan(r)) and torch.equal(torch.isposinf(c), torch.isposinf(r))
    assert torch.equal(torch.isneginf(c), torch.isneginf(r))
    ok = torch.isfinite(r)
    big = r.abs() > 1e30
    assert big[ok].any()
    assert _rel(c[ok & ~big], r[ok & ~big].double()) < _tol(k) and ((c - r).abs() <= 1e-6 * r.abs())[ok & big].all()


@pytest.mark.parametrize("L,P,H,causal", [(68, 68, 8, False), (68, 68, 8, True), (1000, 1000, 64, False), (1000, 1000, 64, True),
                                          (1003, 1004, 20, False), (2052, 2052, 12, False), (2052, 2052, 12, True)])
def test_position_products(L, P, H, causal):
    """The attention's three kinds of product on the matrix-core kernel at sizes that a call may leave to the GEMM library as
    well: two heads, padded rows (two-sided only), causal limits that leave operands' halves unread."""
    B, Nh = 2, 2
    gen = torch.Generator(DEV).manual_seed(L)
    x, y = (torch.randn(B, L, Nh, H, generator=gen, device=DEV) for _ in range(2))
    w = torch.randn(B, Nh, L, P, generator=gen, device=DEV)
    w[..., L:] = 0
    if causal:
        w.tril_()
    prod, t = M.ops._position_product, lambda a: a.double().transpose(1, 2).contiguous()
    s = prod((x, 0), (y, 0), (torch.full_like(w, float("nan")), 1), L, L, H, int(causal), 0.5)[..., :L]
    ref = 0.5 * (t(x) @ t(y).transpose(-1, -2).contiguous())
    keep = torch.ones(L, L, dtype=torch.bool, device=DEV).tril() if causal else torch.ones(L, L, dtype=torch.bool, device=DEV)
    assert _rel(s[..., keep], ref[..., keep]) < _tol(H)
    w64 = w[..., :L].double()
    for transposed in (False, True):
        got = prod((w, 1), (x, 0), (torch.full_like(x, float("nan")), 0), L, H, L, (2 + transposed) * causal, a_rows=transposed, b_rows=True)
        want = (w64.transpose(-1, -2).contiguous() if transposed else w64) @ t(x)
        assert _rel(t(got), want) < _tol(L)


@pytest.mark.parametrize("B,L,Nh,H1,H2", [(2, 1024, 1, 32, 64), (1, 2048, 1, 64, 512)])
def test_attention_on_both_kinds_of_product(B, L, Nh, H1, H2):
    """Sizes of which some products run on the matrix-core kernel and the others in the GEMM library: forward and backward
    against 64 bits."""
    gen = torch.Generator(DEV).manual_seed(L)
    q, k, v, g = (torch.randn(B, L, Nh, h, generator=gen, device=DEV) for h in (H1, H1, H2, H2))
    pays = M.ops._product_pays
    assert len({pays(L, L, H1, B, Nh, 1, False), pays(L, H1, L, B, Nh, 2, False)}) == 2
    y, w = M.ops.attention_fwd(q, k, v, 0.2, 0.0, True, need_weights=True)
    got = M.ops.attention_bwd(g, q, k, v, w, 0.2, True)
    t = [x.double().transpose(1, 2).contiguous().requires_grad_() for x in (q, k, v)]
    s = (0.2 * (t[0] @ t[1].transpose(-1, -2))).masked_fill(torch.ones(L, L, dtype=torch.bool, device=DEV).triu(1), float("-inf"))
    ref = s.softmax(-1) @ t[2]
    ref.backward(g.double().transpose(1, 2))
    assert _rel(y.transpose(1, 2), ref) < 4e-6
    for x, r in zip(got, t):
        assert _rel(x.transpose(1, 2), r.grad) < 1e-5


# sizes on wide tiles: 256 x 128 with every remainder and whole; the same in parts; 256 x 256 all in parts, whole ones and the
# last in parts, with remainders and whole
_WIDE = [(1096, 4360, 1032), (2048, 2048, 1024), (1032, 1048, 8200), (4352, 1032, 8200), (8712, 2056, 4104), (6144, 2816, 1024)]


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("ka,kb", [(0, 0), (0, 1), (1, 0), (1, 1)])
@pytest.mark.parametrize("m,n,k", _WIDE + [(1032, 1048, 8199)])
def test_16bit_products_on_wide_tiles(dtype, ka, kb, m, n, k):
    """As test_16bit_products; columns beside the operands' own hold NaN, and the last rows and columns are checked apart."""
    if k % 8 and not (ka and kb):
        pytest.skip("rows of whole 16-byte pieces")
    print(f"case {dtype} m={m} n={n} k={k} ka={ka} kb={kb}", flush=True)
    gen = torch.Generator(DEV).manual_seed(m + n + k)

    def mk(r, c):
        t = torch.full((r, c + 8), float("nan"), device=DEV, dtype=dtype)
        t[:, :c] = torch.randn(r, c, generator=gen, device=DEV)
        return t[:, :c]

    a, b = mk(k, m) if ka else mk(m, k), mk(k, n) if kb else mk(n, k)
    r = (a.double().t() if ka else a.double()) @ (b.double() if kb else b.double().t())
    c = _gemm(a, b, ka, kb)
    tol = (2.0 ** -9 if dtype is torch.bfloat16 else 2.0 ** -12) + _tol(k)
    assert _rel(c, r) < tol and _rel(c[-8:], r[-8:]) < tol and _rel(c[:, -8:], r[:, -8:]) < tol


@pytest.mark.parametrize("bias,res,silu,pre", [(1, 0, 0, 0), (0, 1, 0, 0), (1, 0, 1, 0), (1, 1, 1, 1), (0, 0, 1, 1), (1, 0, 0, 1)])
@pytest.mark.parametrize("m,n,k", [(1096, 4360, 1032), (1032, 1048, 8200), (6144, 2816, 1024)])
@pytest.mark.parametrize("dtype,ka,kb", [(torch.bfloat16, 0, 0), (torch.float16, 0, 0), (torch.bfloat16, 0, 1), (torch.float16, 1, 1)])
def test_16bit_epilogues_on_wide_tiles(dtype, ka, kb, m, n, k, bias, res, silu, pre):
    """Every way a value is finished, whole tiles and edges, in both types and three orders; with a residual also into the
    residual's own memory."""
    gen = torch.Generator(DEV).manual_seed(8)
    mk = lambda *s: torch.randn(*s, generator=gen, device=DEV).to(dtype)
    a, b, v, x = mk(m, k), mk(n, k), mk(n) * 30, mk(m, n) * 30
    r = a.double() @ b.double().t() + bias * v.double() + res * x.double()
    a, b = a.t().contiguous() if ka else a, b.t().contiguous() if kb else b
    got = _gemm(a, b, ka, kb, v if bias else None, x if res else None, bool(silu), bool(pre))
    c, p = got if pre else (got, None)
    half = 2.0 ** -9 if dtype is torch.bfloat16 else 2.0 ** -12
    tol = half + _tol(k)
    if pre:
        assert _rel(p, r) < tol
    # silu of the rounded value (known where it is written as well; its slope is at most 1.1), rounded again
    assert _rel(c, F.silu(p.double() if pre else r) if silu else r) < (half + 2.0 ** -22 if pre and silu else 3 * tol if silu else tol)
    if res and not pre:
        _call(a, b, x, ka, kb, v if bias else None, x, bool(silu))
        assert torch.equal(x, c)


def test_16bit_workspace_too_small():
    """Wide tiles in parts refuse a workspace that does not hold them, and write nothing."""
    m, n, k = 1032, 1048, 8200
    lib, need = M._lib.load(), M._lib.load().mega_gemm16_workspace_bytes(m, n, k)
    a, b, c = torch.ones(m, k, device=DEV, dtype=torch.bfloat16), torch.ones(n, k, device=DEV, dtype=torch.bfloat16), torch.zeros(m, n, device=DEV, dtype=torch.bfloat16)
    ws = torch.empty(need, dtype=torch.uint8, device=DEV)
    g = _Gemm(a.data_ptr(), b.data_ptr(), c.data_ptr(), None, None, None, k, k, n, 0, 0, 0, 0, 0, 0, 0, m, n, k, 1, 1, 0, 0, 0, 0, 1.0, 0)
    for have, at in ((need - 1, ws.data_ptr()), (need, None)):
        assert need > 0 and lib.mega_gemm16(C.byref(g), 1, at, have, torch.cuda.current_stream().cuda_stream) != 0
    torch.cuda.synchronize()
    assert not bool(c.any())


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16])
@pytest.mark.parametrize("n,k", [(8, 8), (256, 1024)])                  # tiles of 64; wide ones
def test_16bit_silu_of_every_value(dtype, n, k):
    """Half a unit in the last place and 32-bit exp's few units (its argument's rounding: 89 of 2^-24), to the end of exp's range:
    from e^126 ln 2 on the reciprocal of 1 + e^-v alone is no normal number (bf16 -88: -5.3e-37)."""
    v = torch.arange(-32768, 32768, device=DEV).to(torch.int16).view(dtype)
    v = torch.where(v.isfinite(), v, 0)
    a, b = torch.zeros(65536, k, device=DEV, dtype=dtype), torch.zeros(n, k, device=DEV, dtype=dtype)
    a[:, 0], b[:, 0] = v, 1
    c, x = _gemm(a, b, 0, 0, silu=True).double(), v.double()[:, None]
    r = x * torch.where(x < 0, x.exp() / (1 + x.exp()), 1 / (1 + (-x).exp()))
    info = torch.finfo(dtype)
    close = (c - r).abs() <= (info.eps / 2 + 100 * 2.0 ** -24) * r.abs() + info.tiny * info.eps / 2
    assert bool((close | ((x < -88.7) & (c == 0))).all())
