"""The q / k map on runs of tokens (gate_glue.hip: gate_qk_run_kernel, gate_qk_bwd_kernel) at the edges of its rules:
one half vector per lane, one, two, wider rows on the general kernel; a partial last chunk, calls shorter than a chunk,
parameters off their 16-byte boundary.  Reference: the formulas in float64."""
import pytest
import torch

import fairseq_apollo_amd as M
from gpu_util import DEV

pytestmark = pytest.mark.gpu
EPS = {torch.float32: 2.0 ** -23, torch.bfloat16: 2.0 ** -8, torch.float16: 2.0 ** -11}


def _map(z, g, b, freqs, heads, chunk):
    """float64: normalise, two affine maps, rotation of feature pairs per head, positions restarting every `chunk`."""
    T, S = z.shape
    zn = z / z.norm(dim=-1, keepdim=True).clamp(min=1e-5)
    ang = (torch.arange(T, device=z.device) % chunk).double()[:, None] * freqs.double().repeat(heads)[None]
    # the kernel forms pos * freq in float32: the angle is off by half an ulp of it at most
    c, s = ang.cos(), ang.sin()
    out = []
    for i in range(2):
        p = zn * g[i] + b[i]
        x, y = p[:, 0::2], p[:, 1::2]
        out.append(torch.stack((x * c - y * s, x * s + y * c), -1).reshape(T, S))
    return out


@pytest.mark.parametrize("dtype", [torch.float32, torch.bfloat16, torch.float16])
@pytest.mark.parametrize("T,S,heads,chunk,skew", [
    (1, 64, 1, 1024, 0), (7, 64, 2, 1024, 0), (37, 128, 1, 8, 0), (4100, 256, 4, 1000, 0), (64, 264, 1, 16, 0),
    (129, 512, 2, 64, 0), (96, 520, 1, 32, 0), (33, 1024, 4, 16, 0), (20, 1032, 1, 8, 0), (96, 256, 1, 32, 1),
    (9, 30, 3, 4, 0)])
def test_qk_map_and_its_gradients(dtype, T, S, heads, chunk, skew):
    gen = torch.Generator(DEV).manual_seed(T * S)
    z = torch.randn(T, S, generator=gen, device=DEV).to(dtype)
    # skew: parameter rows that start one element behind a 16-byte boundary
    par = torch.randn(4 * S + skew, generator=gen, device=DEV)[skew:]
    g, b = par[:2 * S].view(2, S), par[2 * S:].view(2, S)
    freqs = 10000.0 ** (-torch.arange(S // heads // 2, device=DEV).float() * 2 * heads / S)
    zd, gd, bd = (t.double().requires_grad_(True) for t in (z, g, b))
    want = _map(zd, gd, bd, freqs, heads, chunk)
    q, k = M.ops.gate_qk_fwd(z, g, b, freqs, heads, chunk)
    # one rounding of the result; in float32 the angles' rounding, pos 2^-24 rad of a vector of |want|, on top
    bound = 4 * EPS[dtype] + min(chunk, T) * 2.0 ** -23
    for got, ref in zip((q, k), want):
        assert (got.double() - ref).norm() <= bound * ref.norm()
    vec = 16 // z.element_size()
    if S % vec or S > 128 * vec:
        return
    dq, dk = (torch.randn(T, S, generator=gen, device=DEV).to(dtype) for _ in range(2))
    torch.autograd.backward(want, (dq.double(), dk.double()))
    dz, dg, db = M.ops.gate_qk_bwd(dq, dk, z, g, freqs, heads, chunk)
    assert (dz.double() - zd.grad).norm() <= bound * zd.grad.norm() * (2 if T > 1 else 8)
    for got, ref in ((dg, gd.grad), (db, bd.grad)):
        # float32 sums of T rows: rounding grows no faster than T 2^-24 of the summed magnitudes
        assert (got.double() - ref).norm() <= (min(chunk, T) + 32) * 2.0 ** -22 * ref.norm()
