"""One token of every stream with carried state on the composite step (csrc/decode_layer.hip) against the operators one by
one in fp32 with the same (16-bit rounded) weights, which is the route the oracle pins (test_gpu_model.py): logits after
every token, the carried state after the last one, and the composite step is what ran.

Tolerance (root mean square of the difference over that of the result): a logit is reached through about 30 roundings
to the activation type, each uniform with rms 2^-9 / sqrt(3) relative for bf16 (2^-12 / sqrt(3) for fp16); sqrt(30) of
them is 6.2e-3 (7.7e-4); three times that."""
import copy
import types

import pytest
import torch

import fairseq_apollo_amd as M
from gpu_util import DEV

pytestmark = pytest.mark.gpu
TOL = {torch.bfloat16: 1.9e-2, torch.float16: 2.4e-3}


def _model(D, z, h, heads, ffn, chunk, norm_type, dtype, seed):
    args = types.SimpleNamespace(decoder_embed_dim=D, decoder_layers=2, decoder_z_dim=z, decoder_hidden_dim=h,
                                 decoder_n_dim=16, decoder_ffn_embed_dim=ffn, decoder_chunk_size=chunk,
                                 norm_num_groups=4, num_heads=heads, moving_layer="cema", norm_type=norm_type,
                                 layer_scale=norm_type == "rmsnorm")
    torch.manual_seed(seed)
    model = M.MegaDecoderNoCrossAttn(args, 72, torch.nn.Embedding(72, D, padding_idx=1))
    with torch.no_grad():
        for p in model.parameters():
            if not bool(p.any()):
                p.normal_(0, 0.1)
    half = model.to(DEV).to(dtype).eval()
    return half, copy.deepcopy(half).float()


def _rms(a, b):
    a = torch.view_as_real(a) if a.is_complex() else a
    b = torch.view_as_real(b) if b.is_complex() else b
    return float((a.double() - b.double()).norm() / b.double().norm().clamp(min=1e-30))


# streams around the row tiles (16, 32) and the rows normalised in the projection (4); contexts around the positions per
# workgroup (32), the first token, the token that fills the chunk, the one after it; head widths 8, 24, 64; one slab and
# more (hidden / heads > 512), a width of whole 32-element but not 64-element pieces
@pytest.mark.parametrize("dtype,B,D,z,h,heads,ffn,chunk,prompt,norm_type", [
    (torch.bfloat16, 1, 64, 16, 96, 1, 96, 64, 0, "layernorm"),
    (torch.bfloat16, 4, 96, 32, 1056, 1, 160, 64, 30, "rmsnorm"),
    (torch.float16, 5, 96, 48, 96, 2, 96, 64, 62, "layernorm"),
    (torch.bfloat16, 17, 128, 64, 128, 1, 64, 128, 127, "rmsnorm"),
    (torch.float16, 33, 64, 32, 64, 4, 64, 256, 160, "layernorm"),
    (torch.bfloat16, 64, 64, 16, 64, 2, 64, -1, 33, "layernorm"),
])
def test_token_by_token_logits(dtype, B, D, z, h, heads, ffn, chunk, prompt, norm_type):
    half, full = _model(D, z, h, heads, ffn, chunk, norm_type, dtype, 7 + B)
    tokens = torch.randint(2, 72, (B, prompt + 4), device=DEV)
    tokens[0, prompt + 1] = 1                              # a padded token in one stream
    layer = half.layers[0].mega_layer
    ran = []
    step = layer._token_step
    layer._token_step = lambda *a: ran.append(1) or step(*a)
    sa, sb = {}, {}
    with torch.no_grad():
        for a in range(0, prompt, chunk if chunk > 0 else max(prompt, 1)):
            sl = tokens[:, a:min(prompt, a + chunk) if chunk > 0 else prompt]
            half(sl, incremental_state=sa)
            full(sl, incremental_state=sb)
        for t in range(prompt, prompt + 4):
            la, lb = (m(tokens[:, t:t + 1], incremental_state=s)[0] for m, s in ((half, sa), (full, sb)))
            assert la.shape == lb.shape == (B, 1, 72) and la.dtype == dtype
            assert _rms(la, lb) < TOL[dtype], (t, _rms(la, lb))
    assert len(ran) == 4
    for ea, eb in zip(sa.values(), sb.values()):
        assert sorted(ea) == sorted(eb)
        for k in ea:
            assert ea[k].shape == eb[k].shape, k
            if k == "prev_count":
                assert torch.equal(ea[k], eb[k])
            else:
                assert _rms(ea[k], eb[k]) < TOL[dtype], (k, _rms(ea[k], eb[k]))
    assert M.ops.timestep_norm_status() == 0


def test_state_of_an_earlier_token_survives_the_next():
    """Two continuations of one carried state (beam search keeps such a state): the step writes new state tensors, the
    old ones stay, and the second continuation equals the first."""
    half, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 3)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    state = {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=state)
        before = {n: {k: v.clone() for k, v in e.items()} for n, e in state.items()}
        outs = []
        for _ in range(2):
            mine = {n: dict(e) for n, e in state.items()}
            outs.append(half(tokens[:, 19:], incremental_state=mine)[0])
    assert torch.equal(outs[0], outs[1])
    for n, e in state.items():
        for k, v in e.items():
            assert torch.equal(v, before[n][k]), k


@pytest.mark.parametrize("change", ["hook", "subclass", "columns"])
def test_token_of_modules_that_are_not_plain(change):
    """Projections that someone looks at, replaced by a class of their own or stored column by column are called as
    modules: the values of the operators one by one, in the composite's tolerance."""
    half, full = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    calls = []

    class Own(torch.nn.Linear):
        def forward(self, x):
            calls.append(1)
            return super().forward(x)

    # (the feed-forward block's second projection adds its residual in its product: its weight is read everywhere)
    lins = [m for n, m in half.named_modules() if type(m) is torch.nn.Linear and not n.endswith('fc2')]
    for m in [*lins, half.embed_tokens]:
        if change == "hook":
            m.register_forward_hook(lambda *a: calls.append(1))
        elif change == "columns":
            m.weight.data = m.weight.data.t().contiguous().t()
        elif m is not half.embed_tokens:
            m.__class__ = Own
    sa, sb = {}, {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=sa)
        full(tokens[:, :19], incremental_state=sb)
        calls.clear()
        got, want = half(tokens[:, 19:], incremental_state=sa)[0], full(tokens[:, 19:], incremental_state=sb)[0]
    assert len(calls) == {"hook": len(lins) + 1, "subclass": len(lins), "columns": 0}[change]
    assert _rms(got, want) < TOL[torch.bfloat16]


@pytest.mark.parametrize("name,bias", [("fc2", True), ("fc1", False), ("h_proj", True), ("v_proj", False), ("mx_proj", False)])
def test_token_of_other_projections(name, bias):
    """A projection with a bias where the layer's own has none, and without where it has one: the token is that of the
    operators one by one, in the composite's tolerance, and a bias counts."""
    half, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    for layer in half.layers:
        block = layer.nffn if name.startswith("fc") else layer.mega_layer
        old = getattr(block, name)
        new = torch.nn.Linear(old.in_features, old.out_features, bias=bias)
        torch.nn.init.normal_(new.weight, 0, 0.1)
        if bias:
            torch.nn.init.normal_(new.bias, 0, 1.0)
        setattr(block, name, new.to(DEV).to(torch.bfloat16))
    half.eval()
    full = copy.deepcopy(half).float()
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    sa, sb = {}, {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=sa)
        full(tokens[:, :19], incremental_state=sb)
        got, want = half(tokens[:, 19:], incremental_state=sa)[0], full(tokens[:, 19:], incremental_state=sb)[0]
    assert _rms(got, want) < TOL[torch.bfloat16]


@pytest.mark.parametrize("change", ["forward", "global"])
def test_token_of_replaced_forwards(change):
    """A projection, norm or embedding whose `forward` was replaced on the instance (offloading, adapters), and hooks on
    every module of the program: each is called, as the operators one by one call it."""
    half, full = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    sa, sb, calls = {}, {}, []
    seen = [m for n, m in half.named_modules() if type(m) in (torch.nn.Linear, M.layers.LayerNorm) and not n.endswith('fc2')]
    seen.append(half.embed_tokens)
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=sa)
        full(tokens[:, :19], incremental_state=sb)
        want = full(tokens[:, 19:], incremental_state=sb)[0]
        if change == "forward":
            for m in seen:
                m.forward = lambda x, m=m, f=m.forward: calls.append(m) or f(x)
            got = half(tokens[:, 19:], incremental_state=sa)[0]
        else:
            handle = torch.nn.modules.module.register_module_forward_hook(lambda m, *a: calls.append(m))
            try:
                got = half(tokens[:, 19:], incremental_state=sa)[0]
            finally:
                handle.remove()
    assert all(sum(c is m for c in calls) == 1 for m in seen)
    assert _rms(got, want) < TOL[torch.bfloat16]


class Within(torch.nn.Module):
    """A module that holds another one, and has no weight of its own."""

    def __init__(self, inner):
        super().__init__()
        self.inner = inner

    def forward(self, x):
        return self.inner(x)


def test_modules_without_a_weight():
    """Projections, norms and embeddings inside other modules: token by token and slice by slice as the operators one by
    one, and SwiGLU's first two projections in training too."""
    half, full = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    for m in list(half.modules()):
        for name in ('fc1', 'norm', 'v_proj', 'mx_proj', 'h_proj', 'output_projection', 'embed_tokens'):
            old = m._modules.get(name)
            if type(old) in (torch.nn.Linear, torch.nn.Embedding, M.layers.LayerNorm):
                setattr(m, name, Within(old))
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    sa, sb = {}, {}
    with torch.no_grad():
        for a, b in ((0, 19), (19, 20)):
            got, want = half(tokens[:, a:b], incremental_state=sa)[0], full(tokens[:, a:b], incremental_state=sb)[0]
            assert _rms(got, want) < TOL[torch.bfloat16]
    ffn = M.SwiGLU(64, 96).to(DEV)
    x = torch.randn(2, 9, 64, device=DEV)
    want = ffn(x, x)
    ffn.w1, ffn.w3 = Within(ffn.w1), Within(ffn.w3)
    # fp32: sums of 96 products in another order
    assert _rms(ffn(x, x).detach(), want.detach()) < 1e-6
    with torch.no_grad():
        assert _rms(ffn(x, x), want) < 1e-6


def test_carried_state_under_autocast():
    """Autocast picks the type of every operation: one token leaves the state that the operators one by one leave (keys
    in fp32 behind the normalisation), and mixed types are refused as they are there."""
    half, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    state = {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=state)
        other = {n: dict(e) for n, e in state.items()}
        with torch.autocast('cuda', dtype=torch.bfloat16):
            half(tokens[:, 19:], incremental_state=state)
        with torch.autocast('cuda', dtype=torch.float16), pytest.raises(RuntimeError, match="dtype"):
            half(tokens[:, 19:], incremental_state=other)
    keys = [e["prev_key"] for e in state.values() if "prev_key" in e]
    assert len(keys) == 2 and all(k.dtype == torch.float32 for k in keys)


@pytest.mark.parametrize("entry", ["prev_value", "prev_key", "prev_state", "prev_count"])
def test_token_with_state_in_other_storage(entry):
    """Carried state that starts on no 16 bytes (a view of a packed buffer), counts that are every second of a buffer's:
    the token is that of the operators one by one, in the composite's tolerance."""
    half, full = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    state, sb = {}, {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=state)
        full(tokens[:, :19], incremental_state=sb)
        for part in state.values():
            if entry in part:
                t = part[entry]
                part[entry] = t.repeat_interleave(2)[::2] if entry == "prev_count" else \
                    torch.empty(t.numel() + 1, dtype=t.dtype, device=DEV)[1:].view(t.shape).copy_(t)
        got, want = half(tokens[:, 19:], incremental_state=state)[0], full(tokens[:, 19:], incremental_state=sb)[0]
    assert _rms(got, want) < TOL[torch.bfloat16]


def test_token_masks_of_other_shapes_are_refused():
    """A padding mask is [B, 1] for one token, in the layer and in the norm alone."""
    half, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    x = torch.randn(3, 1, 64, device=DEV, dtype=torch.bfloat16)
    for mask in (torch.zeros(3, dtype=torch.bool, device=DEV), torch.zeros(1, 3, dtype=torch.bool, device=DEV)):
        for module in (half.layers[0].mega_layer, half.final_norm):
            with torch.no_grad(), pytest.raises(RuntimeError, match="padding_mask"):
                module(x, mask, incremental_state={})


def test_layers_see_the_general_mask():
    """Layers of a one-token call get the padding mask they get otherwise: [B, 1], bool."""
    half, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    seen = []
    half.layers[0].register_forward_pre_hook(lambda m, a, kw: seen.append(kw["decoder_padding_mask"]), with_kwargs=True)
    tokens = torch.tensor([[3], [1]], device=DEV)
    with torch.no_grad():
        half(tokens, incremental_state={})
    assert len(seen) == 1 and seen[0].dtype == torch.bool and torch.equal(seen[0], tokens.eq(1))


# around the limits of the one-token projection: the same columns for few and for many rows
@pytest.mark.parametrize("rows,vocab,native", [(16, 8192, True), (17, 8192, False), (8, 16500, True), (9, 16500, False)])
def test_output_projection_of_many_columns(rows, vocab, native):
    """The route follows rows x columns; both routes give the product (fp64 of the same rounded operands; one rounding of
    the result, 2^-9 of it, and fp32 sums)."""
    model, _ = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    torch.manual_seed(vocab)
    model.output_projection = torch.nn.Linear(2048, vocab, bias=False).to(DEV).to(torch.bfloat16)
    x = torch.randn(rows, 1, 2048, device=DEV).to(torch.bfloat16)
    assert M.ops.token_linear_pays(rows, vocab, 2048) == native
    with torch.no_grad():
        got = model.output_layer(x)
        want = x.double() @ model.output_projection.weight.double().t()
    assert got.shape == want.shape and _rms(got, want) < 2 ** -9


# positions per workgroup of 64, 128 and 256 with a partial last block and several rounds of keys and values, heads of
# more than 256 features, several slabs of 512 value columns
@pytest.mark.parametrize("B,z,h,heads,prompt", [
    (64, 128, 1024, 16, 171), (64, 128, 1024, 16, 300), (64, 128, 1024, 16, 700), (40, 512, 2176, 1, 130),
    (64, 64, 4096, 8, 300), (1, 1024, 1056, 2, 200)])
def test_token_attention_of_many_positions(B, z, h, heads, prompt):
    """One token behind a long context against the operators one by one in fp32."""
    half, full = _model(64, z, h, heads, 64, -1, "layernorm", torch.bfloat16, 13)
    tokens = torch.randint(2, 72, (B, prompt + 1), device=DEV)
    layer, ran = half.layers[0].mega_layer, []
    step = layer._token_step
    layer._token_step = lambda *a: ran.append(1) or step(*a)
    sa, sb = {}, {}
    with torch.no_grad():
        half(tokens[:, :prompt], incremental_state=sa)
        full(tokens[:, :prompt], incremental_state=sb)
        got, want = half(tokens[:, prompt:], incremental_state=sa)[0], full(tokens[:, prompt:], incremental_state=sb)[0]
    assert ran and _rms(got, want) < TOL[torch.bfloat16]
    for ea, eb in zip(sa.values(), sb.values()):
        for k in ea:
            if k != "prev_count":
                assert ea[k].shape == eb[k].shape and _rms(ea[k], eb[k]) < TOL[torch.bfloat16], k


class Backwards(M.layers.RotaryEmbedding):
    """Turns the other way."""
    turned = 0

    def rotary(self, x, sidx):
        self.turned += 1
        cis = self._freqs_cis(sidx, sidx + x.shape[-2]).conj()
        return torch.view_as_real(torch.view_as_complex(x.float().unflatten(-1, (-1, 2))) * cis).flatten(-2).to(x.dtype)


class Around(Within):
    """A norm inside another module."""
    seen = 0

    def forward(self, *args, **kwargs):
        self.seen += 1
        return self.inner(*args, **kwargs)


@pytest.mark.parametrize("what", ["rotation", "norm"])
def test_replaced_parts_of_a_layer(what):
    """A rotation of its own class, and a norm inside another module: whole chunks behind whole chunks and one token are
    those of the operators one by one, which ask both (the rotation for q and for k)."""
    half, full = _model(64, 16, 64, 2, 64, 64, "layernorm", torch.bfloat16, 5)
    for layer in (*half.layers, *full.layers):
        if what == "rotation":
            layer.mega_layer.rel_pos_bias.__class__ = Backwards
        else:
            layer.mega_layer.norm = Around(layer.mega_layer.norm)
    tokens = torch.randint(2, 72, (3, 129), device=DEV)
    sa, sb = {}, {}
    with torch.no_grad():
        for a, b in ((0, 64), (64, 128), (128, 129)):
            got, want = half(tokens[:, a:b], incremental_state=sa)[0], full(tokens[:, a:b], incremental_state=sb)[0]
            assert _rms(got, want) < TOL[torch.bfloat16]
    for layer in (*half.layers, *full.layers):
        assert layer.mega_layer.rel_pos_bias.turned == 6 if what == "rotation" else layer.mega_layer.norm.seen == 3


@pytest.mark.parametrize("what", ["bias", "weight", "move_act"])
def test_norm_values_that_are_no_parameters(what):
    """A norm's weight or bias kept as a buffer (frozen for good) counts as it does in the operators one by one."""
    half, full = _model(64, 16, 64, 1, 64, 64, "layernorm", torch.bfloat16, 5)
    for layer in (*half.layers, *full.layers):
        norm, name = (layer.mega_layer.move_act, "weight") if what == "move_act" else (layer.nffn.norm, what)
        value = torch.linspace(-3, 3, 64, device=DEV).to(norm.weight.dtype)
        delattr(norm, name)
        norm.register_buffer(name, value)
    tokens = torch.randint(2, 72, (3, 20), device=DEV)
    sa, sb = {}, {}
    with torch.no_grad():
        half(tokens[:, :19], incremental_state=sa)
        full(tokens[:, :19], incremental_state=sb)
        got, want = half(tokens[:, 19:], incremental_state=sa)[0], full(tokens[:, 19:], incremental_state=sb)[0]
    assert _rms(got, want) < TOL[torch.bfloat16]
