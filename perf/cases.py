"""The work a user of this framework has it do, as cases that can be timed and compared.

Encoder forwards through the model classes (dense batches with and without padding masks, packed batches of different
lengths, the shared-layer model, the int8 model) in the element types that are served, and steps of a decoder built from
`MultiHeadedAttention` and `PositionwiseFeedForward`.  There is no backward direction: the framework serves inference.

Shapes are those of the repository's benchmark and tests: 12 layers of hidden 768 / 12 heads / 3072 ("base"), 24 layers
of 1024 / 16 / 4096 ("large").  A model is loaded once and serves every request, so models are made once per
configuration (weights of the magnitude of trained ones, from a fixed seed); what changes from call to call is the batch.
"""
import math
import random

import torch
from torch import nn

import turbotransformers_amd as tt

VOCAB, POSITIONS = 30522, 512
SIZES = {"base": (12, 768, 12, 3072), "large": (24, 1024, 16, 4096)}
DTYPES = {"f16": torch.float16, "bf16": torch.bfloat16, "f32": torch.float32}
ALBERT_EMBEDDING = 128
DECODER_LAYERS = 6


def listed():
    return [
        # one short query of an interactive service: nothing but latency
        {"name": "bert_f16_b1_s10", "kind": "bert", "size": "base", "dtype": "f16", "batch": 1, "seq": 10, "padded": False},
        # one passage in the element type a checkpoint comes in
        {"name": "bert_f32_b1_s128", "kind": "bert", "size": "base", "dtype": "f32", "batch": 1, "seq": 128, "padded": False},
        # one long document, at a length that is a multiple of nothing
        {"name": "bert_f16_b1_s387", "kind": "bert", "size": "base", "dtype": "f16", "batch": 1, "seq": 387, "padded": False},
        # a serving batch padded to its longest request, with the attention mask that goes with it
        {"name": "bert_f16_b20_s100_mask", "kind": "bert", "size": "base", "dtype": "f16", "batch": 20, "seq": 100, "padded": True},
        # the same service without conversion to half precision
        {"name": "bert_f32_b20_s100_mask", "kind": "bert", "size": "base", "dtype": "f32", "batch": 20, "seq": 100, "padded": True},
        # requests of 5 to 500 tokens, packed; every call has its lengths in another order
        {"name": "packed_f16_20_requests", "kind": "packed", "size": "base", "dtype": "f16", "requests": 20, "shortest": 5,
         "longest": 500, "lengths": 0},
        # the model whose layers share one set of weights
        {"name": "albert_f16_b8_s256", "kind": "albert", "size": "base", "dtype": "f16", "batch": 8, "seq": 256, "padded": False},
        # quantised serving
        {"name": "int8_b20_s128", "kind": "int8", "size": "base", "dtype": "f32", "batch": 20, "seq": 128, "padded": False},
        # one step of a translation decoder: eight hypotheses, 40 tokens generated, a 100-token source
        {"name": "decode_f16_b8_past40", "kind": "decode", "size": "base", "dtype": "f16", "batch": 8, "past": 40, "memory": 100,
         "tokens": 1},
        # its first step: a prefix of 33 tokens, nothing cached, the encoder output projected into keys and values
        {"name": "prefill_f32_b8_s33", "kind": "decode", "size": "base", "dtype": "f32", "batch": 8, "past": 0, "memory": 100,
         "tokens": 33},
        # offline throughput: the headline batch
        {"name": "bert_f16_b64_s512", "kind": "bert", "size": "base", "dtype": "f16", "batch": 64, "seq": 512, "padded": False},
        # offline throughput, the largest model and batch
        {"name": "large_bf16_b64_s512", "kind": "bert", "size": "large", "dtype": "bf16", "batch": 64, "seq": 512, "padded": False},
    ]


def _log_int(rng, low, high):
    return min(high, max(low, int(round(math.exp(rng.uniform(math.log(low), math.log(high)))))))


def draw(rng):
    kind = rng.choice(["bert", "bert", "bert", "bert", "packed", "albert", "int8", "decode"])
    case = {"kind": kind, "size": "base"}
    if kind == "bert":
        case["dtype"] = rng.choice(["f16", "f16", "bf16", "f32"])
        case["size"] = "large" if case["dtype"] == "bf16" else "base"
        case["batch"] = _log_int(rng, 1, 20 if case["dtype"] == "f32" else 64)
        case["seq"] = _log_int(rng, 8, 512)
        case["padded"] = rng.random() < 0.5
    elif kind == "packed":
        case["dtype"] = rng.choice(["f16", "f16", "f32"])
        case["requests"] = _log_int(rng, 2, 32)
        case["shortest"] = rng.randint(1, 20)
        case["longest"] = _log_int(rng, 30, 512)
        case["lengths"] = rng.randrange(1000)
    elif kind == "albert":
        case["dtype"] = rng.choice(["f16", "f16", "f32"])
        case["batch"] = _log_int(rng, 1, 16)
        case["seq"] = _log_int(rng, 8, 512)
        case["padded"] = rng.random() < 0.5
    elif kind == "int8":
        case["dtype"] = "f32"
        case["batch"] = _log_int(rng, 1, 32)
        case["seq"] = _log_int(rng, 8, 512)
        case["padded"] = rng.random() < 0.5
    else:
        case["dtype"] = rng.choice(["f16", "f32"])
        first = rng.random() < 0.3
        case["batch"] = _log_int(rng, 1, 64)
        case["past"] = 0 if first else _log_int(rng, 1, 256)
        case["memory"] = _log_int(rng, 8, 256)
        case["tokens"] = _log_int(rng, 1, 64) if first else 1
    return case


# ---------------------------------------------------------------------------------------------------- models ----------
class _Parts(nn.Module):
    """A module made of named parts: the models are taken over by parameter name, no forward of their own is needed."""

    def __init__(self, **parts):
        super().__init__()
        for name, part in parts.items():
            setattr(self, name, part)

    @property
    def device(self):
        return next(self.parameters()).device


class _Config:
    def __init__(self, **fields):
        self.__dict__.update(fields)


def _embeddings(width):
    return _Parts(word_embeddings=nn.Embedding(VOCAB, width), position_embeddings=nn.Embedding(POSITIONS, width),
                  token_type_embeddings=nn.Embedding(2, width), LayerNorm=nn.LayerNorm(width))


def _bert_layer(hidden, heads, ffn):
    proj = _Parts(query=nn.Linear(hidden, hidden), key=nn.Linear(hidden, hidden), value=nn.Linear(hidden, hidden))
    proj.num_attention_heads = heads
    attention = _Parts(output=_Parts(dense=nn.Linear(hidden, hidden), LayerNorm=nn.LayerNorm(hidden)))
    attention.add_module("self", proj)
    return _Parts(attention=attention, intermediate=_Parts(dense=nn.Linear(hidden, ffn)),
                  output=_Parts(dense=nn.Linear(ffn, hidden), LayerNorm=nn.LayerNorm(hidden)))


def _albert_layer(hidden, heads, ffn):
    attention = _Parts(query=nn.Linear(hidden, hidden), key=nn.Linear(hidden, hidden), value=nn.Linear(hidden, hidden),
                       dense=nn.Linear(hidden, hidden), LayerNorm=nn.LayerNorm(hidden))
    attention.num_attention_heads = heads
    return _Parts(attention=attention, ffn=nn.Linear(hidden, ffn), ffn_output=nn.Linear(ffn, hidden),
                  full_layer_layer_norm=nn.LayerNorm(hidden))


def _onmt_attention(hidden, heads):
    attention = _Parts(linear_keys=nn.Linear(hidden, hidden), linear_values=nn.Linear(hidden, hidden),
                       linear_query=nn.Linear(hidden, hidden), final_linear=nn.Linear(hidden, hidden))
    attention.head_count = heads
    return attention


def _onmt_layer(hidden, heads, ffn):
    return _Parts(self_attn=_onmt_attention(hidden, heads), self_norm=nn.LayerNorm(hidden),
                  context_attn=_onmt_attention(hidden, heads), context_norm=nn.LayerNorm(hidden),
                  feed_forward=_Parts(w_1=nn.Linear(hidden, ffn), w_2=nn.Linear(ffn, hidden), layer_norm=nn.LayerNorm(hidden)))


def _with_weights(module, dtype):
    """Matrices N(0, 0.02^2), biases and LayerNorm parameters around 0 and 1 as training leaves them."""
    gen = torch.Generator(device="cuda").manual_seed(1234)
    with torch.no_grad():
        for name, p in module.named_parameters():
            p.normal_(0.0, 0.02, generator=gen)
            if "norm" in name.lower() and name.endswith("weight"):
                p.add_(1.0)
    return module.to(DTYPES[dtype]).eval()


_MODELS = {}


def _model(kind, size, dtype):
    """The loaded model of a configuration: (what serves the calls, the torch module whose weights it uses)."""
    key = (kind, size, dtype)
    if key in _MODELS:
        return _MODELS[key][0]
    layers, hidden, heads, ffn = SIZES[size]
    with torch.device("cuda"):
        if kind in ("bert", "packed", "int8"):
            torch_model = _Parts(embeddings=_embeddings(hidden),
                                 encoder=_Parts(layer=nn.ModuleList(_bert_layer(hidden, heads, ffn) for _ in range(layers))),
                                 pooler=_Parts(dense=nn.Linear(hidden, hidden)))
        elif kind == "albert":
            groups = nn.ModuleList([_Parts(albert_layers=nn.ModuleList([_albert_layer(hidden, heads, ffn)]))])
            torch_model = _Parts(embeddings=_embeddings(ALBERT_EMBEDDING),
                                 encoder=_Parts(embedding_hidden_mapping_in=nn.Linear(ALBERT_EMBEDDING, hidden),
                                                albert_layer_groups=groups),
                                 pooler=nn.Linear(hidden, hidden))
        else:
            torch_model = nn.ModuleList(_onmt_layer(hidden, heads, ffn) for _ in range(DECODER_LAYERS))
    _with_weights(torch_model, dtype)
    torch_model.config = _Config(num_hidden_layers=layers, num_hidden_groups=1, num_attention_heads=heads)
    device = torch.device("cuda:0")
    if kind == "bert":
        served = tt.BertModel.from_torch(torch_model, device, "turbo")
    elif kind == "packed":
        served = tt.BertModelSmartBatch.from_torch(torch_model, device)
    elif kind == "int8":
        served = tt.QBertModel.from_torch(torch_model, backend="turbo")
    elif kind == "albert":
        served = tt.AlbertModel.from_torch(torch_model, device)
    else:
        served = [(tt.MultiHeadedAttention.from_onmt(layer.self_attn, layer.self_norm),
                   tt.MultiHeadedAttention.from_onmt(layer.context_attn, layer.context_norm),
                   tt.PositionwiseFeedForward.from_onmt(layer.feed_forward)) for layer in torch_model]
    _MODELS[key] = (served, torch_model)
    return served


# ---------------------------------------------------------------------------------------------------- passes ----------
def _packed_lengths(case):
    rng = random.Random(case["lengths"])
    return [rng.randint(case["shortest"], case["longest"]) for _ in range(case["requests"])]


def prepare(case, seed):
    state = {"kind": case["kind"], "model": _model(case["kind"], case["size"], case["dtype"])}
    gen = torch.Generator(device="cuda").manual_seed(seed)
    rng = random.Random(seed)

    def ids(*shape):
        return torch.randint(0, VOCAB, shape, generator=gen, device="cuda", dtype=torch.int64)

    if case["kind"] == "packed":
        lens = _packed_lengths(case)
        rng.shuffle(lens)
        state.update(lens=lens, ids=[ids(1, n) for n in lens])
    elif case["kind"] == "decode":
        _, hidden, heads, _ = SIZES[case["size"]]
        b, past, d = case["batch"], case["past"], hidden // heads

        def values(*shape):
            return torch.randn(shape, generator=gen, device="cuda").to(DTYPES[case["dtype"]])

        state["x"], state["memory"] = values(b, case["tokens"], hidden), values(b, case["memory"], hidden)
        state["caches"] = [
            {"memory_keys": values(b, heads, case["memory"], d) if past else None,
             "memory_values": values(b, heads, case["memory"], d) if past else None,
             "self_keys": values(b, heads, past, d) if past else None,
             "self_values": values(b, heads, past, d) if past else None} for _ in range(DECODER_LAYERS)]
        # source positions past a hypothesis' own sentence are masked; a prefix does not look ahead
        source = torch.tensor([rng.randint((case["memory"] + 1) // 2, case["memory"]) for _ in range(b)], device="cuda")
        columns = torch.arange(case["memory"], device="cuda")
        state["source_mask"] = (columns[None, None, :] >= source[:, None, None]).float() * -1e18
        t = case["tokens"]
        state["self_mask"] = None if past else torch.triu(torch.full((t, t), -1e18, device="cuda"), 1).repeat(b, 1, 1)
    else:
        b, s = case["batch"], case["seq"]
        state["ids"], state["mask"] = ids(b, s), None
        if case["padded"]:
            lens = torch.tensor([s] + [rng.randint((s + 2) // 3, s) for _ in range(b - 1)], device="cuda")
            state["mask"] = (torch.arange(s, device="cuda")[None, :] < lens[:, None]).long()
    return state


def run(state):
    model, kind = state["model"], state["kind"]
    if kind == "packed":
        return model(state["ids"], state["lens"])
    if kind == "decode":
        x, grown, attn = state["x"], [], None
        for (self_attn, context_attn, feed_forward), cache in zip(model, state["caches"]):
            cache = dict(cache)
            x, _ = self_attn(x, x, x, state["self_mask"], cache, "self", pre_layernorm=True, post_add_input=True)
            x, attn = context_attn(state["memory"], state["memory"], x, state["source_mask"], cache, "context",
                                   pre_layernorm=True, post_add_input=True)
            x = feed_forward(x)
            grown.append(cache)
        return {"hidden": x, "attention": attn, "caches": grown}
    if kind == "bert":
        return model(state["ids"], attention_masks=state["mask"])
    return model(state["ids"], state["mask"])


def work(case):
    layers, hidden, heads, ffn = SIZES[case["size"]]
    e = 2 if case["dtype"] in ("f16", "bf16") else 4
    if case["kind"] == "decode":
        b, t, past, memory = case["batch"], case["tokens"], case["past"], case["memory"]
        rows, keys = b * t, past + t
        weights = 6 * hidden * hidden + 2 * hidden * ffn
        flops = 2 * rows * weights + 4 * rows * hidden * (keys + memory)
        cache_io = 2 * b * hidden * (past + keys) + 2 * b * hidden * memory
        if past == 0:
            weights += 2 * hidden * hidden
            flops += 4 * b * memory * hidden * hidden
        outputs = rows * hidden + rows * heads * memory / DECODER_LAYERS
        return {"bytes": e * (DECODER_LAYERS * (weights + cache_io + outputs) + rows * hidden), "flops": DECODER_LAYERS * flops}
    lens = _packed_lengths(case) if case["kind"] == "packed" else [case["seq"]] * case["batch"]
    tokens, pooled = sum(lens), 1 if case["kind"] == "packed" else len(lens)
    per_layer = 4 * hidden * hidden + 2 * hidden * ffn
    flops = layers * (2 * tokens * per_layer + 4 * hidden * sum(n * n for n in lens)) + 2 * pooled * hidden * hidden
    matrices = per_layer * (1 if case["kind"] == "albert" else layers)
    matrix_bytes = matrices * (1 if case["kind"] == "int8" else e) + hidden * hidden * e
    embedding = ALBERT_EMBEDDING if case["kind"] == "albert" else hidden
    if case["kind"] == "albert":
        flops += 2 * tokens * embedding * hidden
    return {"bytes": matrix_bytes + 8 * tokens + e * (tokens * (embedding + hidden) + pooled * hidden), "flops": flops}


def tolerance(case):
    if case["kind"] == "int8":
        # a value next to a rounding boundary may land on either side: one step of 1/127 of the largest value
        return {"rel": 1e-2}
    # f32: sums of up to 3072 products in another order, through the layers; f16 / bf16: roundings of the stored
    # activations and of the attention probabilities, through the layers
    return {"rel": {"f32": 3e-5, "f16": 5e-3, "bf16": 1e-2}[case["dtype"]]}
