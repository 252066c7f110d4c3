"""The calls this framework is timed on: what a user's program has it do, through the public entry points.

`listed()` names twelve of them, `draw(rng)` gives more of the same ranges.  A case is a dict of plain values; its
"kind" selects how `prepare` builds what a program holds before the call (modules with their weights, inputs, carried
state) and what `run` does with it once:

    token          one token of every stream through a language model with carried state (generation)
    recurrent      one token of every stream through the fused norm -> moving average decode step
    prefill        logits of whole token sequences (any length: the model pads to whole chunks)
    stream         logits of documents taken slice by slice with carried state (validation of long documents)
    lm_train       loss and gradients of a language model
    encoder_train  loss and gradients of two-sided encoder layers on padded batches
    average        one moving-average layer on rows in time
    block          TimestepNorm -> moving average, the head of every layer
    block_train    the same forwards and backwards
    layer          one Mega2 layer forwards
    layer_train    one Mega2 layer forwards and backwards

Weights start from the modules' own initialisation; what that sets to zero or one (norm weights, biases, the q / k
map) is moved off it, as the first training steps do."""
import math
import types

import torch
import torch.nn.functional as F

import fairseq_apollo_amd as M

DEV = "cuda:0"
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
VOCAB = 264                       # bytes and special symbols: character-level language modelling
STATES = 16                       # moving-average states per channel
PAD = 1


def listed():
    return [
        # interactive generation: one stream, in the middle of a chunk; the smallest call there is, all launches
        {"name": "token_b1", "kind": "token", "dtype": "bf16", "batch": 1, "context": 700, "dim": 1024, "heads": 1,
         "chunk": 1024},
        # streaming decode of many streams at once, 64 streams of 2048 channels
        {"name": "recurrent_b64", "kind": "recurrent", "dtype": "bf16", "batch": 64, "dim": 2048},
        # prompts of a length that is not a whole number of chunks (the last one is padded)
        {"name": "prefill_ragged", "kind": "prefill", "dtype": "bf16", "batch": 2, "length": 2991, "dim": 1024,
         "heads": 2, "chunk": 1024},
        # perplexity of long documents in single precision, slice by slice
        {"name": "stream_fp32", "kind": "stream", "dtype": "fp32", "batch": 2, "length": 3072, "dim": 512, "heads": 1,
         "chunk": 1024},
        # a language model's training step at an ordinary size, single head
        {"name": "lm_train", "kind": "lm_train", "dtype": "bf16", "batch": 4, "length": 2048, "dim": 1024, "heads": 1,
         "chunk": 1024},
        # classification of byte sequences: two-sided layers, padded batch, single precision
        {"name": "encoder_train", "kind": "encoder_train", "dtype": "fp32", "batch": 8, "length": 1000, "dim": 256,
         "layer": "cema"},
        # a long two-sided real moving average in single precision with a right-padding mask
        {"name": "average_two_sided", "kind": "average", "dtype": "fp32", "batch": 1, "length": 16384, "dim": 256,
         "layer": "ema", "two_sided": True, "mask": True},
        # the head of a layer at the headline size
        {"name": "block_headline", "kind": "block", "dtype": "bf16", "batch": 4, "length": 4096, "dim": 1024,
         "mask": False},
        # the same path off its best shape: 48-channel norm groups, an odd length, padding, fp16
        {"name": "block_ragged", "kind": "block", "dtype": "fp16", "batch": 3, "length": 1501, "dim": 768, "mask": True},
        # what the head of a layer costs in training, at the headline size
        {"name": "block_train", "kind": "block_train", "dtype": "bf16", "batch": 4, "length": 4096, "dim": 1024,
         "mask": False},
        # one whole layer over a long sequence: four chunks of 2048, four heads
        {"name": "layer_forward", "kind": "layer", "dtype": "bf16", "batch": 1, "length": 8192, "dim": 2048, "heads": 4,
         "chunk": 2048},
        # its training step, the largest call
        {"name": "layer_train", "kind": "layer_train", "dtype": "bf16", "batch": 1, "length": 8192, "dim": 2048,
         "heads": 4, "chunk": 2048},
    ]


def draw(rng):
    def spread(low, high):            # whole numbers even over their logarithm, odd ones among them
        return int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))

    kind = rng.choice(["token", "recurrent", "prefill", "stream", "lm_train", "encoder_train", "average", "block", "block",
                       "block_train", "layer", "layer_train"])
    half = rng.choice(["bf16", "bf16", "fp16"])
    if kind == "token":
        return {"kind": kind, "dtype": half, "batch": spread(1, 48), "context": spread(16, 3000),
                "dim": rng.choice([512, 768, 1024]), "heads": rng.choice([1, 2, 4]), "chunk": rng.choice([512, 1024])}
    if kind == "recurrent":
        return {"kind": kind, "dtype": rng.choice(["bf16", "fp16", "fp32"]), "batch": spread(1, 128),
                "dim": rng.choice([512, 1024, 1536, 2048])}
    if kind in ("prefill", "lm_train"):
        batch = spread(1, 8)
        return {"kind": kind, "dtype": "bf16" if kind == "lm_train" else half, "batch": batch,
                "length": spread(100, 8192 // batch), "dim": rng.choice([512, 768, 1024]), "heads": rng.choice([1, 2, 4]),
                "chunk": rng.choice([512, 1024])}
    if kind == "stream":
        chunk, batch = rng.choice([256, 512, 1024]), spread(1, 4)
        return {"kind": kind, "dtype": rng.choice(["fp32", "bf16"]), "batch": batch,
                "length": chunk * rng.randint(1, 4), "dim": rng.choice([256, 512, 768]), "heads": rng.choice([1, 2]),
                "chunk": chunk}
    if kind == "encoder_train":
        length = spread(128, 2048)
        return {"kind": kind, "dtype": "fp32", "batch": spread(1, max(2, 8192 // length)), "length": length,
                "dim": rng.choice([128, 256, 512]), "layer": rng.choice(["ema", "cema"])}
    if kind == "average":
        length = spread(256, 16384)
        return {"kind": kind, "dtype": rng.choice(["fp32", "fp16", "bf16"]), "batch": spread(1, max(2, 32768 // length)),
                "length": length, "dim": rng.choice([128, 256, 512, 1024]), "layer": rng.choice(["ema", "cema"]),
                "two_sided": rng.random() < 0.5, "mask": rng.random() < 0.5}
    if kind in ("block", "block_train"):
        length = spread(64, 8192)
        return {"kind": kind, "dtype": rng.choice(["bf16", "bf16", "fp16", "fp32"]),
                "batch": spread(1, max(2, 16384 // length)), "length": length,
                "dim": rng.choice([512, 768, 1024, 1536, 2048]), "mask": rng.random() < 0.5}
    chunk = rng.choice([512, 1024, 2048])
    length = chunk * rng.randint(1, 8192 // chunk)
    return {"kind": kind, "dtype": half if kind == "layer" else "bf16", "batch": spread(1, max(1, 8192 // length)),
            "length": length, "dim": rng.choice([1024, 2048]), "heads": rng.choice([1, 2, 4]), "chunk": chunk}


def _sizes(dim):
    """(z, hidden, feed-forward) widths of a layer of `dim` channels: a quarter, twice and eleven quarters of it."""
    return dim // 4, 2 * dim, dim * 11 // 4


def _settle(module, gen):
    """Parameters that start at zero leave it; the generator is on the device."""
    with torch.no_grad():
        for p in module.parameters():
            if not bool(p.any()):
                p.normal_(0.0, 0.1, generator=gen)
    return module


def _language_model(case):
    z, hidden, ffn = _sizes(case["dim"])
    args = types.SimpleNamespace(
        decoder_embed_dim=case["dim"], decoder_layers=2, decoder_z_dim=z, decoder_hidden_dim=hidden, decoder_n_dim=STATES,
        decoder_ffn_embed_dim=ffn, decoder_chunk_size=case["chunk"], norm_num_groups=16, num_heads=case["heads"],
        moving_layer="cema")
    return M.MegaDecoderNoCrossAttn(args, VOCAB, torch.nn.Embedding(VOCAB, case["dim"], padding_idx=PAD))


def _encoder(case):
    dim = case["dim"]
    args = types.SimpleNamespace(
        encoder_embed_dim=dim, encoder_z_dim=dim // 4, encoder_hidden_dim=2 * dim, encoder_n_dim=STATES,
        encoder_ffn_embed_dim=2 * dim, encoder_chunk_size=-1, norm_num_groups=16, moving_layer=case["layer"],
        max_source_positions=2048)
    return torch.nn.ModuleList([M.MegaEncoderLayer(args) for _ in range(2)])


def _padding(batch, length, gen):
    """Right padding of up to a quarter of every row."""
    kept = length - torch.randint(0, length // 4 + 1, (batch, 1), generator=gen, device=DEV)
    return torch.arange(length, device=DEV)[None, :] >= kept


def prepare(case, seed):
    kind, dtype = case["kind"], DTYPES[case["dtype"]]
    torch.manual_seed(seed)
    gen = torch.Generator(DEV).manual_seed(seed)

    def normal(*shape):
        return torch.randn(*shape, generator=gen, device=DEV).to(dtype)

    def tokens(*shape):
        return torch.randint(4, VOCAB, shape, generator=gen, device=DEV)

    s = {"kind": kind}
    if kind in ("token", "prefill", "stream", "lm_train"):
        model = _settle(_language_model(case).to(DEV), gen).to(dtype)
        s["model"] = model.train() if kind == "lm_train" else model.eval()
        if kind == "token":
            prompt, carried = tokens(case["batch"], case["context"]), {}
            with torch.no_grad():
                for a in range(0, case["context"], case["chunk"]):
                    model(prompt[:, a:a + case["chunk"]], incremental_state=carried)
            s["carried"], s["tokens"] = carried, tokens(case["batch"], 1)
        else:
            s["tokens"] = tokens(case["batch"], case["length"])
        if kind == "lm_train":
            s["target"] = tokens(case["batch"], case["length"])
    elif kind == "recurrent":
        ema = _settle(M.MultiHeadComplexEMA(case["dim"], ndim=STATES).to(DEV), gen).eval()
        p, q, g = ema.coeffs()
        s["step"] = M.ops.DecodeStep(torch.randn(case["dim"], generator=gen, device=DEV) * 0.1,
                                     torch.randn(case["dim"], generator=gen, device=DEV) * 0.1, 16, 1e-5, p.squeeze(-1),
                                     q.squeeze(-1), g, ema.omega.detach().reshape(-1), case["batch"])
        for _ in range(4):                     # streams that are under way
            s["step"](normal(case["batch"], case["dim"]))
        s["x"] = normal(case["batch"], case["dim"])
    elif kind == "encoder_train":
        s["layers"] = _settle(_encoder(case).to(DEV), gen).to(dtype).train()
        s["x"] = normal(case["batch"], case["length"], case["dim"]).requires_grad_(True)
        s["weight"] = normal(case["batch"], case["length"], case["dim"])
        s["mask"] = _padding(case["batch"], case["length"], gen)
    elif kind == "average":
        cls = M.MultiHeadEMA if case["layer"] == "ema" else M.MultiHeadComplexEMA
        s["layer"] = _settle(cls(case["dim"], ndim=STATES, bidirectional=case["two_sided"]).to(DEV), gen).eval()
        s["x"] = normal(case["batch"], case["dim"], case["length"])
        s["mask"] = _padding(case["batch"], case["length"], gen) if case["mask"] else None
    elif kind in ("block", "block_train"):
        s["norm"] = _settle(M.TimestepNorm(case["dim"], 16).to(DEV), gen).train(kind == "block_train")
        s["move"] = M.MultiHeadComplexEMA(case["dim"], ndim=STATES).to(DEV).train(kind == "block_train")
        s["x"] = normal(case["batch"], case["length"], case["dim"])
        s["mask"] = _padding(case["batch"], case["length"], gen) if case["mask"] else None
        if kind == "block_train":
            s["x"].requires_grad_(True)
            s["grads"] = (normal(case["batch"], case["length"], case["dim"]),
                          normal(case["batch"], case["length"], case["dim"]))
    else:
        z, hidden, ffn = _sizes(case["dim"])
        layer = M.Mega2Layer(case["dim"], z, hidden, STATES, ffn, case["chunk"], norm_num_groups=16,
                             num_heads=case["heads"], moving_act="silu")
        layer = _settle(layer.to(DEV), gen).to(dtype)
        s["layer"] = layer.train(kind == "layer_train")
        s["x"] = normal(case["batch"], case["length"], case["dim"])
        if kind == "layer_train":
            s["x"].requires_grad_(True)
            s["weight"] = normal(case["batch"], case["length"], case["dim"])
    return s


def _gradients(module, x=None):
    got = [p.grad for p in module.parameters()]
    return got if x is None else [x.grad] + got


def _clear(module, x=None):
    module.zero_grad(set_to_none=True)
    if x is not None:
        x.grad = None


def run(s):
    kind = s["kind"]
    if kind == "token":
        # the streams' state stays with the caller (as beam search keeps it): the call gets a dictionary of its own
        carried = {name: dict(entry) for name, entry in s["carried"].items()}
        with torch.no_grad():
            logits, _ = s["model"](s["tokens"], incremental_state=carried)
        state = [entry[k] for entry in carried.values()
                 for k in ("prev_count", "prev_mean", "prev_var", "prev_state", "prev_key", "prev_value") if k in entry]
        return [logits] + state
    if kind == "recurrent":
        with torch.no_grad():
            xn, y = s["step"](s["x"])
        return [xn, y, s["step"].state]
    if kind == "prefill":
        with torch.no_grad():
            return s["model"](s["tokens"])[0]
    if kind == "stream":
        with torch.no_grad():
            return s["model"].streamed(s["tokens"])
    if kind == "lm_train":
        _clear(s["model"])
        logits, _ = s["model"](s["tokens"])
        loss = F.cross_entropy(logits.float().view(-1, VOCAB), s["target"].view(-1))
        loss.backward()
        return [loss.detach(), logits.detach()] + _gradients(s["model"])
    if kind == "encoder_train":
        _clear(s["layers"], s["x"])
        x = s["x"]
        for layer in s["layers"]:
            x = layer(x, s["mask"])
        (x * s["weight"]).sum().backward()
        return [x.detach()] + _gradients(s["layers"], s["x"])
    if kind == "average":
        with torch.no_grad():
            return s["layer"](s["x"], s["mask"])
    if kind == "block":
        with torch.no_grad():
            return M.norm_then_move(s["norm"], s["move"], s["x"], s["mask"], out_layout="input")
    if kind == "block_train":
        for module in (s["norm"], s["move"]):
            module.zero_grad(set_to_none=True)
        s["x"].grad = None
        xn, y = M.norm_then_move(s["norm"], s["move"], s["x"], s["mask"], out_layout="input")
        torch.autograd.backward((xn, y.transpose(1, 2)), s["grads"])
        return [xn.detach(), y.detach(), s["x"].grad] + _gradients(s["norm"]) + _gradients(s["move"])
    if kind == "layer":
        with torch.no_grad():
            return s["layer"](s["x"])
    _clear(s["layer"], s["x"])
    y = s["layer"](s["x"])
    (y * s["weight"]).sum().backward()
    return [y.detach()] + _gradients(s["layer"], s["x"])


def _attention_flops(pairs, z, hidden):
    """The two products over `pairs` (query, key) pairs that the mask lets through, all heads together."""
    return 2 * pairs * (z + hidden)


def work(case):
    kind, es, d = case["kind"], 4 if case["dtype"] == "fp32" else 2, case["dim"]
    b, n = case["batch"], case.get("length", 1)
    tok = b * n
    ema = 8 * STATES                                        # one complex multiply-add per state each way in and out
    if kind == "recurrent":
        return {"bytes": 2 * b * d * STATES * 8 + 3 * b * d * es, "flops": b * d * 2 * ema}
    if kind == "average":
        return {"bytes": 2 * tok * d * es + (tok if case["mask"] else 0),
                "flops": tok * d * ema * (2 if case["two_sided"] else 1)}
    if kind == "block":
        return {"bytes": 3 * tok * d * es + (tok if case["mask"] else 0), "flops": tok * d * (ema + 8)}
    if kind == "block_train":
        # forwards x in, xn and y out; backwards x and both gradients in, the gradient of x out
        return {"bytes": 7 * tok * d * es + (tok if case["mask"] else 0), "flops": tok * d * 3 * (ema + 8)}
    z, hidden, ffn = _sizes(d)
    attn_w = d * hidden + d * (z + hidden + 2 * d) + hidden * d
    if kind == "encoder_train":
        z, hidden, ffn = d // 4, 2 * d, 2 * d
        weights = 2 * (d * hidden + d * (z + hidden + 2 * d) + hidden * d + 2 * d * ffn)
        fwd = 2 * tok * weights + 2 * (_attention_flops(b * n * n, z, hidden) + tok * d * 2 * ema)
        return {"bytes": 2 * weights * es + 4 * tok * d * es, "flops": 3 * fwd}
    if kind in ("layer", "layer_train"):
        weights = attn_w + 3 * d * ffn
        chunk = min(case["chunk"], n)
        fwd = 2 * tok * weights + _attention_flops(tok * (chunk + 1) // 2, z, hidden) + tok * d * ema
        if kind == "layer":
            return {"bytes": weights * es + 2 * tok * d * es, "flops": fwd}
        return {"bytes": 2 * weights * es + 4 * tok * d * es, "flops": 3 * fwd}
    weights = 2 * (attn_w + 2 * d * ffn) + d * VOCAB        # two layers and the output projection
    if kind == "token":
        seen = case["context"] % case["chunk"] + 1
        state = 2 * (2 * b * d * STATES * 8 + b * (z + hidden) * (2 * seen - 1) * es)
        return {"bytes": weights * es + state + b * VOCAB * es,
                "flops": b * (2 * weights + 2 * (_attention_flops(seen, z, hidden) + d * ema))}
    chunk = min(case["chunk"], n)
    fwd = 2 * tok * weights + 2 * (_attention_flops(tok * (chunk + 1) // 2, z, hidden) + tok * d * ema)
    io = tok * 8 + tok * VOCAB * es
    if kind == "lm_train":
        return {"bytes": 2 * weights * es + io, "flops": 3 * fwd}
    return {"bytes": weights * es + io, "flops": fwd}


# Largest relative error of any output against the same path in 64 bits, over the listed and some forty drawn cases,
# times four: one operator or two (forwards 2.4e-3, 3e-4, 2.1e-7; with gradients 2.8e-3, 3.5e-4, 2.1e-6), whole models
# and layers (forwards 4.7e-3, 5.8e-4, 4.6e-7; with gradients 1.2e-2 and 1.6e-2, -, 5.4e-6; held to 3e-2).
TOLERANCE = {
    ("operator", False): {"bf16": 1e-2, "fp16": 1.2e-3, "fp32": 1e-6},
    ("operator", True): {"bf16": 1.1e-2, "fp16": 1.4e-3, "fp32": 8e-6},
    ("model", False): {"bf16": 2e-2, "fp16": 2.3e-3, "fp32": 2e-6},
    ("model", True): {"bf16": 3e-2, "fp16": 4e-3, "fp32": 2e-5},
}


def tolerance(case):
    part = "operator" if case["kind"] in ("recurrent", "average", "block", "block_train") else "model"
    return {"rel": TOLERANCE[part, case["kind"].endswith("train")][case["dtype"]]}
