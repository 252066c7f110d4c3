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


def test_norm_widths():
    """What the gates of the norms and of the feed-forward composites ask: parameters as wide as the rows."""
    for norm in (M.layers.LayerNorm(8), M.layers.RMSNorm(8)):
        assert M.modules.norm_width_ok(norm, 8) and not M.modules.norm_width_ok(norm, 16)
    assert not M.modules.norm_width_ok(M.layers.LayerNorm(8, elementwise_affine=False), 16)
    with pytest.raises(RuntimeError):
        M.layers.LayerNorm(8, elementwise_affine=False)(torch.zeros(2, 16))
