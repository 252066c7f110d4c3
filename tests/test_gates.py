"""Rules that send a call to a fused operator instead of the modules' own calls: what they must leave alone.  No GPU: the
rules only look at modules and shapes (where a rule asks for device tensors, that question is answered for it)."""
import types

import pytest
import torch

import fairseq_apollo_amd as M
from fairseq_apollo_amd import layers


def _two_sided(**kw):
    return M.MovingAverageGatedAttention(16, 8, 32, 4, norm_num_groups=4, bidirectional=True, **kw)


def _padded(layer, monkeypatch):
    """Whether attention with padded keys would run as the one fused operator (shapes and types taken as fitting)."""
    monkeypatch.setattr(M.ops, "own_attention_products", lambda *a: True)
    q, v = torch.zeros(2, 64, 1, 8), torch.zeros(2, 64, 1, 32)
    return layer._padded_product(q, q, v, torch.zeros(2, 64, dtype=torch.bool))


class _OwnBias(layers.SimpleRelativePositionalBias):
    pass


@pytest.mark.parametrize("bias,fused", [(None, True), (layers.SimpleRelativePositionalBias, False), (_OwnBias, False)])
def test_padded_attention_adds_every_learned_bias(bias, fused, monkeypatch):
    """A learned bias, of the class itself or one derived from it, belongs to the scores: the fused operator has none."""
    layer = _two_sided()
    if bias is not None:
        layer.rel_pos_bias = bias(64)
    assert _padded(layer, monkeypatch) == fused


@pytest.mark.parametrize("layer_trains,softmax_trains,fused", [(False, False, True), (True, True, False), (False, True, False),
                                                               (True, False, True)])
def test_padded_attention_drops_what_its_softmax_drops(layer_trains, softmax_trains, fused, monkeypatch):
    """Dropped keys follow the softmax module's own mode (sampling with dropout keeps the layer in eval mode)."""
    layer = _two_sided(attention_dropout=0.5).train(layer_trains)
    layer.attn_softmax.train(softmax_trains)
    assert layer.attn_softmax._dropout > 0
    assert _padded(layer, monkeypatch) == fused


def _language_model():
    args = types.SimpleNamespace(decoder_embed_dim=16, decoder_layers=2, decoder_z_dim=8, decoder_hidden_dim=32, decoder_n_dim=4,
                                 decoder_ffn_embed_dim=16, decoder_chunk_size=8, norm_num_groups=4, moving_layer="cema")
    return M.MegaDecoderNoCrossAttn(args, 32, torch.nn.Embedding(32, 16, padding_idx=1)).eval()


_ON_DEVICE = types.SimpleNamespace(is_cuda=True)


def test_replaced_final_norm_keeps_the_general_path():
    """A norm of another kind (no groups to speak of) in the place of the last one: its output is cleared at padding."""
    model = _language_model()
    with torch.no_grad():
        assert model._norm_clears(_ON_DEVICE) and model._mask_stays(_ON_DEVICE)
        model.final_norm = torch.nn.LayerNorm(16)
        assert not model._norm_clears(_ON_DEVICE) and not model._mask_stays(_ON_DEVICE)


class _Other(torch.nn.Module):
    """A layer's part with its call's signature and nothing else."""

    def forward(self, x, *args, **kw):
        return x


@pytest.mark.parametrize("part", ["", "norm", "move"])
def test_replaced_parts_of_a_layer_get_no_mask_of_zeros(part):
    """The mask of a call without padding goes to the layers only where every module that receives it is the package's
    own, unwatched: another one keeps getting None."""
    model = _language_model()
    layer = model.layers[1]
    with torch.no_grad():
        if part:
            hook = getattr(layer.mega_layer, part).register_forward_pre_hook(lambda m, i: None)
            assert not model._mask_stays(_ON_DEVICE)
            hook.remove()
            assert model._mask_stays(_ON_DEVICE)
            setattr(layer.mega_layer, part, _Other())
        else:
            layer.mega_layer = _Other()
        assert not model._mask_stays(_ON_DEVICE)


def test_scripted_linear_layers_run_as_they_are():
    lin, x = torch.nn.Linear(16, 8), torch.randn(3, 5, 16)
    with torch.no_grad():
        assert torch.equal(M.modules.project(torch.jit.script(lin), x), lin(x))


class _Scripted(torch.nn.Module):
    def forward(self, x):
        return x + 1


def test_scripted_layers_get_no_mask_of_zeros():
    """A scripted module among the layers, or in a layer's place for its attention: the mask rule says no."""
    model = _language_model()
    with torch.no_grad():
        model.layers[1] = torch.jit.script(_Scripted())
        assert not model._mask_stays(_ON_DEVICE)
        model.layers[1] = _language_model().layers[1]
        model.layers[1].mega_layer = torch.jit.script(_Scripted())
        assert not model._mask_stays(_ON_DEVICE)
