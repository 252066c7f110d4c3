"""What the native host code (csrc/host.cpp) refuses before anything is launched, and the rules of the modules that send
calls there.  No GPU: the operands lie in host memory, every check comes before the launch."""
import pytest
import torch

import fairseq_apollo_amd as M

H = M._lib.load_host()
RMS, LN = M.ops.TOKEN_RMSNORM, M.ops.TOKEN_LAYERNORM


@pytest.mark.parametrize("call", [
    lambda x, w: H.row_norm_forward(x, RMS, w, None, 1e-5, 0),
    lambda x, w: H.row_norm_forward(x, LN, None, w, 1e-5, 0),
    lambda x, w: H.row_norm_backward(x, x, RMS, w, None, 1e-5, 0),
    lambda x, w: H.row_norm_backward(x, x, LN, None, w, 1e-5, 0),
    lambda x, w: H.ffn_forward(x, LN, w, w, 1e-5, torch.zeros(16, 8), torch.zeros(16), torch.zeros(8, 16), 0),
], ids=["forward weight", "forward bias", "backward weight", "backward bias", "feed-forward"])
@pytest.mark.parametrize("width", [4, 16])
def test_row_norm_parameters_of_another_width(call, width):
    """Kernels take the width from the rows: parameters of another width would be read, and their gradients written,
    out of range."""
    with pytest.raises(RuntimeError, match="norm parameters of %d values on rows of 8" % width):
        call(torch.zeros(2, 8), torch.zeros(width))


def test_composite_operands_of_other_shapes():
    D, S, E = 8, 4, 16
    x, mx = torch.zeros(1, 3, D), torch.zeros(1, D, 3)
    W = 2 * D + S + E
    good = [x, mx, torch.zeros(E, D), torch.zeros(E), torch.zeros(W, D), torch.zeros(W), torch.zeros(2, S), torch.zeros(2, S),
            torch.zeros(S // 2), 1, 3, RMS, torch.zeros(D), 1e-5, 0]
    for i, bad in ((4, torch.zeros(W - 1, D)), (7, torch.zeros(2, S + 2)), (12, torch.zeros(D - 1))):
        args = list(good)
        args[i] = bad
        with pytest.raises(RuntimeError, match="mix_forward: argument %d must be" % i):
            H.mix_forward(*args)
    with pytest.raises(RuntimeError, match="mix_out_forward: argument 1 must be"):
        H.mix_out_forward(x, torch.zeros(3, W + 2), torch.zeros(3, E), torch.zeros(D, E), S, 0)
    with pytest.raises(RuntimeError, match="mix_out_forward: argument 3 must be"):
        H.mix_out_forward(x, torch.zeros(3, W), torch.zeros(3, E), torch.zeros(D - 2, E), S, 0)
    with pytest.raises(RuntimeError, match="swiglu_forward: argument 3 must be"):
        H.swiglu_forward(x[0], None, torch.zeros(12, D), torch.zeros(8, D), torch.zeros(D, 12), 0)


def test_backward_operands_of_other_shapes():
    """The backward passes size their kernels from a saved operand or two: the others must fit."""
    D, S, E, T = 8, 4, 16, 3
    W = 2 * D + S + E
    x, row = torch.zeros(1, T, D), lambda *s: torch.zeros(*s)
    out = [x, x, row(T, W), row(T, E), row(T, E), row(T, D), row(D, E), S, 0, 15]
    for i, bad in ((0, row(1, T, D - 1)), (2, row(T, W + 2)), (3, row(T - 1, E)), (4, row(T, E - 2)), (5, row(T, E)), (6, row(D + 1, E))):
        args = list(out)
        args[i] = bad
        with pytest.raises(RuntimeError, match="mix_out_backward: "):
            H.mix_out_backward(*args)
    back = [row(T, S), row(T, S), row(T, E), row(T, W), x, row(T, E), x, x, row(T, W), row(E, D), row(W, D), row(2, S), row(S // 2),
            1, T, RMS, row(D), 1e-5, 0, 1023]
    for i, bad in ((0, row(T, S + 2)), (2, row(T + 1, E)), (3, row(T, W + 1)), (6, row(1, T, D + 8)), (8, row(T + 1, W)),
                   (10, row(W, D - 1)), (11, row(2, S + 2)), (16, row(D + 8))):
        args = list(back)
        args[i] = bad
        with pytest.raises(RuntimeError, match="mix_backward: "):
            H.mix_backward(*args)
    ffn = [x, x, x, row(T, 6), row(T, 6), LN, row(D), row(D), 1e-5, row(6, D), row(D, 6), 0, 63]
    for i, bad in ((0, row(1, T + 1, D)), (3, row(T, 5)), (4, row(T + 1, 6))):
        args = list(ffn)
        args[i] = bad
        with pytest.raises(RuntimeError, match="ffn_backward: "):
            H.ffn_backward(*args)
    with pytest.raises(RuntimeError, match="swiglu_backward: argument 3 must be"):
        H.swiglu_backward(x, x, row(T, 6), row(T, 5), row(T, 6), row(6, D), row(6, D), row(D, 6), 0, 31)


def test_norm_widths():
    """What the gates of the norms and of the feed-forward composites ask: parameters as wide as the rows."""
    for norm in (M.layers.LayerNorm(8), M.layers.RMSNorm(8)):
        assert M.modules.norm_width_ok(norm, 8) and not M.modules.norm_width_ok(norm, 16)
    assert not M.modules.norm_width_ok(M.layers.LayerNorm(8, elementwise_affine=False), 16)
    with pytest.raises(RuntimeError):
        M.layers.LayerNorm(8, elementwise_affine=False)(torch.zeros(2, 16))


@pytest.mark.parametrize("scale,pad", [(8.0, 1), (None, None)])
def test_token_embedding(scale, pad):
    """The one-token step's lookup is torch's: the scaled rows and the mask that the general path forms, and an index
    outside the table is refused as torch refuses it."""
    table = torch.randn(7, 8, dtype=torch.bfloat16)
    tokens = torch.tensor([[3], [1], [6]])
    x, mask = H.token_embed(tokens, table, scale, pad)
    want = torch.nn.functional.embedding(tokens, table)
    assert torch.equal(x, want if scale is None else scale * want)
    assert mask is None if pad is None else torch.equal(mask, tokens.eq(pad))
    for bad in (7, -1):
        with pytest.raises(RuntimeError):
            H.token_embed(torch.tensor([[bad]]), table, scale, pad)


@pytest.mark.parametrize("native", [True, False])
def test_tensor_versions(native, monkeypatch):
    """The key of the eval-mode caches: any number of tensors, with the native library and (modules on the CPU) without;
    an edit in place and another storage change it."""
    if not native:
        monkeypatch.setattr(M._lib, "_host", None)
        monkeypatch.setattr(M._lib, "HOST_PATH", M._lib.HOST_PATH + ".none")
    m = torch.nn.Module()
    for i in range(80):
        m.register_parameter(f"p{i}", torch.nn.Parameter(torch.zeros(2)) if i != 40 else None)
    keys = [M.modules._tensor_versions(m)]
    assert M.modules._tensor_versions(m) == keys[0]
    with torch.no_grad():
        m.p79.add_(1)
    keys.append(M.modules._tensor_versions(m))
    m.p0.data = torch.zeros(2)
    keys.append(M.modules._tensor_versions(m))
    assert len(set(keys)) == 3
    layer = M.MultiHeadComplexEMA(8, ndim=4).eval()
    p, q, g = layer.coeffs()
    with torch.no_grad():
        layer.alpha.add_(1.0)
    assert not torch.equal(layer.coeffs()[0], p)


def test_composites_leave_the_interpreter_to_other_threads():
    """A composite's work runs without the interpreter lock: another thread goes on under a long product (in host memory;
    the weight of the next product does not fit, so the call ends before anything is launched)."""
    import threading
    import time

    ticks, stop = [], threading.Event()

    def count():
        while not stop.is_set():
            ticks.append(time.perf_counter())
            time.sleep(0.001)

    T, D, N = 40000, 512, 512
    args = [torch.randn(T, D), torch.randn(T, D), *(torch.randn(T, N) for _ in range(3)), torch.randn(N, D), torch.randn(N, D),
            torch.randn(D + 1, N), 0, 31]
    threads = torch.get_num_threads()
    torch.set_num_threads(1)
    other = threading.Thread(target=count)
    other.start()
    try:
        begin = time.perf_counter()
        with pytest.raises(RuntimeError):
            H.swiglu_backward(*args)
        end = time.perf_counter()
    finally:
        stop.set()
        other.join()
        torch.set_num_threads(threads)
    # about one a millisecond; with the lock held none but at the edges
    assert sum(begin < t < end for t in ticks) > 100 * (end - begin)


@pytest.mark.parametrize("cpg", [32, 48, 64, 96, 128])
@pytest.mark.parametrize("dtype", [0, 1, 2])
def test_sizes_of_the_one_kernel_pair(dtype, cpg):
    """TimestepNorm -> moving average in one launch (dtype: 0 fp32, 1 bf16, 2 fp16): not where the two operators are more
    accurate, which short rows are and, behind a partial block, the state handed on; bf16 in whole lines always was."""
    one = lambda L, state=0, rows=False: M.ops.norm_ema_one_kernel(dtype, 2, L, 4 * cpg, 4, 16, state, rows)
    always = dtype == 1 and cpg in (64, 128)
    shortest = 256 if dtype == 1 else 64
    assert one(2048) and one(2048, 3) and one(1000) and one(1000, 0, True) and one(1024, 2) and one(shortest)
    assert one(shortest - 1) == one(1) == one(1000, 2) == one(2049, 2) == always
    assert not one(1000, 1) and not one(1000, 3) and not one(1001, 0, True)
    assert one(16 * 1024) and not one(16 * 1024, 1) and not one(17 * 1024)
    assert not M.ops.norm_ema_one_kernel(dtype, 2, 2048, 4 * 24, 4, 16, 0, False)


@pytest.mark.parametrize("m,n,k,gradient,own", [
    (8000, 512, 256, 0, 1), (2048, 2176, 512, 0, 1), (16384, 2048, 1024, 0, 1), (4096, 4096, 2048, 0, 1), (1, 128, 128, 0, 1),
    (300, 2048, 1024, 0, 1), (512, 256, 8000, 1, 1), (1088, 256, 8000, 1, 1), (512, 2048, 4096, 0, 0), (1000, 1024, 4352, 0, 0),
    (2048, 1024, 2816, 0, 0), (2048, 512, 1024, 0, 1), (2048, 1024, 1024, 0, 1), (1024, 1024, 8000, 1, 0), (2048, 1024, 8000, 1, 0), (512, 512, 16384, 0, 0), (512, 512, 16384, 1, 1), (1, 16384, 4096, 0, 0)])
def test_sizes_of_the_fp32_products(m, n, k, gradient, own):
    """fp32 products that the matrix-core kernel serves clearly slower than the GEMM library are left to it."""
    assert M._lib.load().mega_gemm_f32_pays(m, n, k, gradient, gradient) == own


def test_the_limit_of_16bit_products_stands_once():
    """modules.own_product asks no native call beyond the size at which mega_gemm16_pays says no."""
    flops, (m, n) = M.modules.OWN_16BIT_FLOPS, (1000, 1000)
    k = int(flops / (2 * m * n))
    assert M._lib.load().mega_gemm16_pays(m, n, k, 0, 0) == 1 and M._lib.load().mega_gemm16_pays(m, n, k + 1, 0, 0) == 0


@pytest.mark.parametrize("m,n,k,order,silu,own", [
    (2048, 4096, 1024, 0, 0, 1), (5000, 2048, 1024, 0, 0, 0), (4096, 2816, 1024, 0, 0, 1), (4096, 2048, 4096, 0, 0, 0), (8192, 2816, 1024, 0, 0, 0), (8192, 2048, 5632, 0, 0, 0), (8192, 8192, 8192, 0, 0, 0),
    (8192, 4096, 2048, 0, 0, 0), (32768, 5632, 2048, 0, 0, 0), (12000, 2816, 1024, 0, 0, 1), (8192, 5632, 2048, 0, 0, 1), (16384, 8704, 2048, 0, 0, 0),
    (8192, 3264, 768, 0, 0, 1), (65536, 2056, 2048, 0, 0, 0), (5000, 2048, 1024, 0, 1, 1), (8192, 4096, 2048, 0, 1, 1),
    (8192, 4096, 8192, 0, 1, 0), (2048, 512, 8192, 0, 1, 1), (1 << 29, 136, 8, 0, 1, 0), (8192, 2048, 5632, 1, 0, 1), (8192, 8192, 8192, 3, 0, 1)])
def test_sizes_of_the_16bit_products(m, n, k, order, silu, own):
    """x W^T that the device computes clearly faster in the GEMM library, where the device and not its call's host time is the
    bound, is left to it; with silu, whose pass the library's product does not spare, and the gradients' orders are not."""
    lib = M._lib.load()
    assert (lib.mega_gemm16_silu_pays if silu else lib.mega_gemm16_pays)(m, n, k, order >> 1, order & 1) == own


@pytest.mark.parametrize("m,n,k,own", [((1 << 30) - 64, 8, 8, 1), (1 << 30, 8, 8, 0), (8, 1 << 30, 8, 0), ((1 << 29) - 64, 128, 8, 1), (1 << 29, 136, 8, 0)])
@pytest.mark.parametrize("a_kmajor,b_kmajor", [(0, 1), (1, 1)])
def test_16bit_products_that_no_launch_takes(m, n, k, own, a_kmajor, b_kmajor):
    """Sizes beyond the kernels' 32 bits or a launch's 2^32 threads are left to the GEMM library, not refused."""
    assert M._lib.load().mega_gemm16_pays(m, n, k, a_kmajor, b_kmajor) == own


@pytest.mark.parametrize("m,n,k,batch,heads,causal,a_kmajor,own", [
    (512, 512, 128, 8, 1, 0, 0, 1), (1000, 64, 1000, 8, 1, 0, 0, 0), (4096, 64, 4096, 2, 1, 2, 0, 0), (512, 512, 1024, 1, 1, 1, 0, 0),
    (1000, 1000, 64, 16, 4, 0, 0, 1), (2048, 2048, 1024, 4, 1, 0, 0, 1), (2048, 2048, 32, 8, 1, 0, 0, 0), (1000, 1000, 512, 8, 1, 0, 0, 1),
    (2048, 2048, 512, 2, 1, 0, 0, 0), (2048, 1024, 2048, 2, 1, 3, 1, 1), (64, 2048, 64, 64, 1, 2, 0, 0), (2048, 64, 2048, 1, 1, 0, 0, 1), (1024, 1024, 1024, 2, 1, 2, 0, 1),
    (2048, 128, 2048, 8, 1, 0, 0, 0)])
def test_sizes_of_the_fp32_attention_products(m, n, k, batch, heads, causal, a_kmajor, own):
    """Batched fp32 products that the matrix-core kernel serves clearly slower than the GEMM library are left to it."""
    assert M._lib.load().mega_gemm_f32_batched_pays(m, n, k, batch, heads, causal, a_kmajor) == own


@pytest.mark.parametrize("m,n,k,parts", [(600, 1024, 2816, 0), (1000, 1024, 2816, 0), (768, 768, 2048, 0), (1000, 768, 3264, 0), (1000, 2048, 4096, 1), (300, 2048, 4096, 1)])
def test_16bit_products_in_parts(m, n, k, parts):
    """One workgroup of 64 x 64 on every compute unit is not taken for half of two: wide tiles in parts, and their second
    launch, only where they are the quicker ones."""
    assert (M._lib.load().mega_gemm16_workspace_bytes(m, n, k) > 0) == parts
