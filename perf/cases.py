"""Timed cases of the quantized-Linear paths, as a program that serves a quantized model calls them.

Four kinds of pass (a case's ``op``):

* ``linears``: the quantized Linears of ``layers`` decoder layers of one architecture on ``tokens`` rows, through the
  modules (E8-D4 q|k|v and gate|up as ``EPTQMultiLinear``, everything else as ``EPTQLinear``).  Decode batches run as
  a decode step does, captured once in a HIP graph and replayed (``graph``); prompts and the small OPT model run the
  modules eagerly, as a model from ``load_quantized_model`` does.
* ``dequant``: ``EPTQLinear.dequantize`` of the same Linears.
* ``prompt``: ``QuantLlama.forward_tokens`` of whole prompts, logits out.
* ``step``: one captured ``QuantLlama.decode_next`` step after a prompt, logits out.

Weights, scales and activations follow ``eptq_amd.synthetic``: indices uniform over the codebook, a per-mille or so of
critical blocks, log-normal column scales, unit normal activations (a decoder's normalized hidden states).
"""

import functools
import math

import torch
import torch.nn.functional as F

from eptq_amd.kernels import decode_workspace
from eptq_amd.kernels.linear import EPTQLinear, EPTQMultiLinear
from eptq_amd.llama import GraphDecoder, LlamaConfig, build_synthetic
from eptq_amd.quantizers import E8D4Quantizer, E8LatticeQuantizer
from eptq_amd.synthetic import make_layer

DEV = "cuda"

# Per architecture: the groups of Linears that read one input, each (in_features, [out_features, ...]), and whether
# the Linears carry a bias.
FAMILIES = {
    "opt125m": ([(768, [768, 768, 768]), (768, [768]), (768, [3072]), (3072, [768])], True),
    "llama2_7b": ([(4096, [4096, 4096, 4096]), (4096, [4096]), (4096, [11008, 11008]), (11008, [4096])], False),
    "llama2_13b": ([(5120, [5120, 5120, 5120]), (5120, [5120]), (5120, [13824, 13824]), (13824, [5120])], False),
    "llama3_8b": ([(4096, [4096, 1024, 1024]), (4096, [4096]), (4096, [14336, 14336]), (14336, [4096])], False),
}
RADIUS = {"e8_d4": 1.75, "e8_lattice": 1.6}


def _linears(name, family, tokens, **more):
    case = {"name": name, "op": "linears", "family": family, "quantizer": "e8_d4", "layers": 1, "tokens": tokens,
            "dtype": "float16", "group": 0, "percmask": 0.002, "graph": False}
    case.update(more)
    return case


def listed():
    return [
        # Interactive use of a small model: one token through one OPT-125m layer on the default E8 lattice, eager
        # modules with biases; call overhead and launches are what a user waits for.
        _linears("opt125m_e8_token", "opt125m", 1, quantizer="e8_lattice"),
        # Single-user decoding, the framework's headline: a token's Linears, cold weights (more than the caches hold).
        _linears("llama2_7b_decode_b1", "llama2_7b", 1, layers=8, percmask=0.001, graph=True),
        # The same for a small serving batch, and for a larger one of a grouped bf16 model.
        _linears("llama2_7b_decode_b8", "llama2_7b", 8, layers=8, percmask=0.001, graph=True),
        _linears("llama3_8b_group_bf16_decode_b16", "llama3_8b", 16, layers=8, group=128, dtype="bfloat16", graph=True),
        # A full serving batch: 64 sequences decoded together (or one short chunk of a prompt).
        _linears("llama2_7b_decode_b64", "llama2_7b", 64, layers=6, percmask=0.001, graph=True),
        # A small batch of an E8-lattice model, whose table does not fit the LDS.
        _linears("llama2_7b_e8_decode_b4", "llama2_7b", 4, layers=4, quantizer="e8_lattice", graph=True),
        # A chat-sized prompt, and a long one of a larger model.
        _linears("llama2_7b_prompt_512", "llama2_7b", 512, layers=2, percmask=0.001),
        _linears("llama2_13b_prompt_2048", "llama2_13b", 2048),
        # A grouped bf16 model's prompt of no special length.
        _linears("llama3_8b_group_bf16_prompt_1000", "llama3_8b", 1000, group=128, dtype="bfloat16"),
        # Reconstruction of a layer's fp16 weights (export, merging, comparison with the unquantized model).
        dict(_linears("llama2_7b_dequantize", "llama2_7b", 0, percmask=0.01), op="dequant"),
        # Whole calls: the prompts of two sequences, and one greedy step after a prompt.
        {"name": "llama_prompt_logits", "op": "prompt", "hidden": 4096, "ffn": 11008, "heads": 32, "kv_heads": 32,
         "vocab": 32000, "layers": 2, "batch": 2, "context": 500},
        {"name": "llama_step_logits", "op": "step", "hidden": 4096, "ffn": 11008, "heads": 32, "kv_heads": 32,
         "vocab": 32000, "layers": 8, "batch": 1, "context": 500},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.random()
    if kind < 0.12:
        heads = rng.choice([16, 32])
        batch = rng.choice([1, 1, 2, 4, 8])
        return {"op": rng.choice(["prompt", "step"]), "hidden": 128 * heads, "ffn": 64 * rng.randint(80, 172),
                "heads": heads, "kv_heads": rng.choice([heads, heads // 4]), "vocab": rng.choice([16000, 32000]),
                "layers": rng.randint(1, 2), "batch": batch, "context": _log_int(rng, 16, 1000 // batch)}
    case = {"op": "dequant" if kind < 0.22 else "linears", "family": rng.choice(sorted(FAMILIES)),
            "quantizer": rng.choice(["e8_d4", "e8_d4", "e8_lattice"]), "layers": 1,
            "tokens": _log_int(rng, 1, 2048), "dtype": rng.choice(["float16", "float16", "bfloat16"]),
            "group": rng.choice([0, 0, 128]), "percmask": round(math.exp(rng.uniform(math.log(5e-4), math.log(1e-2))), 5),
            "graph": False}
    if case["op"] == "dequant":
        case.update(tokens=0, dtype="float16")
    elif kind > 0.85:
        # A Linear of no particular model: features in whole 8s only (no group), few tokens.
        case.update(family="%dx%d" % (8 * _log_int(rng, 32, 512), 8 * _log_int(rng, 32, 512)), group=0,
                    tokens=_log_int(rng, 1, 100))
    case["graph"] = 0 < case["tokens"] <= 128 and rng.random() < 0.7
    return case


def _groups(case):
    if case["family"] in FAMILIES:
        return FAMILIES[case["family"]]
    out, inp = (int(v) for v in case["family"].split("x"))
    return [(inp, [out])], True


@functools.lru_cache(maxsize=None)
def _quantizer(kind):
    """The loaded codebook a program keeps for all of its layers."""
    return (E8D4Quantizer if kind == "e8_d4" else E8LatticeQuantizer)(device=DEV, radius=RADIUS[kind])


def _captured(fn):
    side = torch.cuda.Stream()
    side.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(side):
        fn()
    torch.cuda.current_stream().wait_stream(side)
    torch.cuda.synchronize()
    graph = torch.cuda.CUDAGraph()
    with torch.cuda.graph(graph):
        out = fn()
    return graph, out


def _config(case):
    return LlamaConfig(hidden=case["hidden"], ffn=case["ffn"], layers=case["layers"], heads=case["heads"],
                       kv_heads=case["kv_heads"], vocab=case["vocab"])


@torch.no_grad()
def prepare(case, seed):
    gen = torch.Generator(device=DEV).manual_seed(seed)
    if case["op"] in ("prompt", "step"):
        model = build_synthetic(_config(case), device=DEV, seed=seed)
        for layer in model.layers:  # trained models' norm weights lie well below 1, and their attention is not one-hot
            layer.input_layernorm.weight.mul_(0.3)
            layer.post_attention_layernorm.weight.mul_(0.3)
        ids = torch.randint(0, case["vocab"], (case["batch"], case["context"] + 1), generator=gen, device=DEV)
        dec = GraphDecoder(model, case["batch"], case["context"] + 16, device=DEV)
        state = {"case": case, "model": model, "dec": dec, "ids": ids}
        if case["op"] == "prompt":
            state["pos"] = torch.arange(case["context"], device=DEV)
            return state
        dec.prefill(ids[:, :-1].contiguous())
        last = ids[:, -1:].contiguous()

        def step():     # the same step each time: the token and its position are set before it
            torch.add(last, 0, out=dec.tok)
            dec.pos.fill_(case["context"])
            return model.decode_next(dec.tok, dec.pos)

        state["graph"], state["logits"] = _captured(step)
        return state

    groups, biased = _groups(case)
    q = _quantizer(case["quantizer"])
    work = decode_workspace(DEV) if case["graph"] else None
    dtype = getattr(torch, case["dtype"])
    mods, xs, k = [], [], 0
    for _ in range(case["layers"]):
        for inp, outs in groups:
            lins = []
            for out in outs:
                qd = make_layer(out, inp, seed=seed * 1009 + k, percmask=case["percmask"], bias=biased,
                                qb_size=case["group"] or None, device=DEV)
                lins.append(EPTQLinear.from_quantized_data(qd, q, case["quantizer"]).to(DEV))
                k += 1
            fused = case["quantizer"] == "e8_d4" and len(lins) > 1 and case["op"] == "linears"
            x = torch.randn((case["tokens"], inp), generator=gen, device=DEV).to(dtype)
            for m in [EPTQMultiLinear(lins)] if fused else lins:
                m._work = work
                mods.append(m)
                xs.append(x)
    state = {"case": case, "mods": mods, "xs": xs}
    if case["graph"]:
        state["graph"], state["ys"] = _captured(lambda: [m(x) for m, x in zip(mods, xs)])
    return state


@torch.no_grad()
def run(state):
    op = state["case"]["op"]
    if op == "prompt":
        return state["model"].forward_tokens(state["ids"][:, :-1], state["pos"])
    if op == "step":
        state["graph"].replay()
        return state["logits"]
    if op == "dequant":
        return [m.dequantize() for m in state["mods"]]
    if "graph" in state:
        state["graph"].replay()
        return state["ys"]
    return [m(x) for m, x in zip(state["mods"], state["xs"])]


def _linear_work(out, inp, case):
    """Bytes of one Linear's indices, scales and critical blocks (the table is shared and small)."""
    M = out // 8
    nnz = round(case["percmask"] * M * inp)
    b = 2 * M * inp + 20 * nnz + 4 * (M + 1) + 2 * out + 2 * inp
    return b + (2 * (out // case["group"]) * inp if case["group"] else 0)


def work(case):
    if case["op"] in ("prompt", "step"):
        h, f, b, t = case["hidden"], case["ffn"], case["batch"], case["context"]
        kv = case["kv_heads"] * (h // case["heads"])
        shapes = [(h, h), (kv, h), (kv, h), (h, h), (f, h), (f, h), (h, f)]
        like = {"percmask": 0.002, "group": 0}
        rows = b * (t if case["op"] == "prompt" else 1)
        n_bytes = case["layers"] * sum(_linear_work(o, i, like) for o, i in shapes) + 2 * case["vocab"] * h
        flops = 2.0 * rows * (case["layers"] * sum(o * i for o, i in shapes) + case["vocab"] * h)
        pairs = b * (t * (t + 1) // 2 if case["op"] == "prompt" else t + 1)
        flops += case["layers"] * 4.0 * pairs * h
        n_bytes += case["layers"] * 4 * b * kv * (t + 1) + 2 * rows * case["vocab"]
        return {"bytes": n_bytes, "flops": flops}
    groups, biased = _groups(case)
    n_bytes, flops = 0, 0.0
    for inp, outs in groups:
        for out in outs:
            n_bytes += _linear_work(out, inp, case)
            if case["op"] == "dequant":
                n_bytes += 2 * out * inp
                flops += 2.0 * out * inp
            else:
                n_bytes += 2 * case["tokens"] * out + (2 * out if biased else 0)
                flops += 2.0 * case["tokens"] * out * inp
        n_bytes += 2 * case["tokens"] * inp
    return {"bytes": case["layers"] * n_bytes, "flops": case["layers"] * flops}


def tolerance(case):
    # About four times the error against 64 bits: 2e-4 to 5e-4 in fp16 (rounded activations and outputs), 1.7e-3 in
    # bf16; whole models, where a rounding travels on, 4e-4 to 3e-3.
    if case["op"] == "dequant":
        return "exact"
    if case["op"] in ("prompt", "step"):
        return {"rel": 1e-2}
    return {"rel": 7e-3 if case["dtype"] == "bfloat16" else 2e-3}


def _dense(lin, table):
    """A layer's weights in 64 bits: table vectors times group scales, critical blocks, row and column scales."""
    Q = lin.Q.long()
    M, N = Q.shape
    u = Q + 32768
    tab = table.double()
    if lin.quantizer_type == "e8_d4":
        a = tab[(u >> 7).clamp(max=511)]
        b = tab[((u >> 14) << 7) | (u & 127)]
        v = torch.cat((a, b), dim=-1)
    else:
        v = tab[u.clamp(max=65534)]
    w = v.permute(0, 2, 1).reshape(8 * M, N)
    if lin.S_group is not None:
        S = lin.S_group.double()
        w = w * S.repeat_interleave(8 * M // S.shape[0], dim=0)
    m, n = (Q == 32767).nonzero(as_tuple=True)
    if m.numel():
        w = w.reshape(M, 8, N)
        w[m, :, n] = lin.O_vals.double()
        w = w.reshape(8 * M, N)
    return w.mul_(lin.g.double()[:, None]).mul_(lin.h.double()[None, :])


def _apply(mod, x):
    parts = list(mod.parts) if isinstance(mod, EPTQMultiLinear) else [mod]
    ys = []
    for p in parts:
        y = x @ _dense(p, p._codebook).t()
        ys.append(y if p.bias is None else y + p.bias.double())
    return torch.cat(ys, dim=-1)


def _exact_logits(model, ids, cfg):
    """The model in 64 bits on whole sequences: logits (B, T, vocab)."""
    B, T = ids.shape
    H, Hk, D = cfg.heads, cfg.kv_heads, cfg.head_dim
    inv = 1.0 / (cfg.rope_theta ** (torch.arange(0, D, 2, device=DEV).double() / D))
    ang = torch.outer(torch.arange(T, device=DEV).double(), inv)
    cos, sin = torch.cat((ang, ang), -1).cos(), torch.cat((ang, ang), -1).sin()

    def norm(x, n):
        return x * torch.rsqrt(x.pow(2).mean(-1, keepdim=True) + cfg.eps) * n.weight.double()

    def rope(t):
        a, b = t[..., :D // 2], t[..., D // 2:]
        return t * cos + torch.cat((-b, a), -1) * sin

    x = model.embed_tokens.weight.double()[ids]
    mask = torch.full((T, T), float("-inf"), dtype=torch.float64, device=DEV).triu(1)
    for layer in model.layers:
        qkv = _apply(layer.qkv_proj, norm(x, layer.input_layernorm))
        q, k, v = (t.reshape(B, T, -1, D).transpose(1, 2) for t in qkv.split([H * D, Hk * D, Hk * D], dim=-1))
        q, k = rope(q), rope(k).repeat_interleave(H // Hk, dim=1)
        v = v.repeat_interleave(H // Hk, dim=1)
        p = torch.softmax(torch.matmul(q, k.transpose(-1, -2).contiguous()) / math.sqrt(D) + mask, dim=-1)
        x = x + _apply(layer.o_proj, torch.matmul(p, v.contiguous()).transpose(1, 2).reshape(B, T, H * D))
        gate, up = _apply(layer.gate_up_proj, norm(x, layer.post_attention_layernorm)).chunk(2, dim=-1)
        x = x + _apply(layer.down_proj, F.silu(gate) * up)
    return norm(x, model.norm) @ model.lm_head.weight.double().t()


@torch.no_grad()
def exact(case, seed):
    state = prepare(case, seed)
    if case["op"] == "prompt":
        return _exact_logits(state["model"], state["ids"][:, :-1], _config(case))
    if case["op"] == "step":
        return _exact_logits(state["model"], state["ids"], _config(case))[:, -1]
    if case["op"] == "dequant":
        return [_dense(m, m._table_f32) for m in state["mods"]]
    return [_apply(m, x.double()) for m, x in zip(state["mods"], state["xs"])]
