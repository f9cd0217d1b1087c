"""What a user of this library has it do, as cases that can be timed and checked.

Six kinds of work, each through the library's public entry points:

  layer    one decoder layer of a decode step (``mk_lib.decode_step`` with hidden states)
  step     a whole decode step, logits and greedy tokens (``NeuronLlamaForCausalLM.forward``)
  loop     greedy generation in one launch (``mk_lib.decode_loop``)
  first    a prompt up to its first token's logits (``NeuronLlamaForCausalLM.prefill`` and a decode step)
  prefill  one decoder layer of context encoding (``mk_lib.prefill`` with the hidden state out)
  sample   the next tokens from logits (``mk_lib.sample``)

Weights are the library's own synthetic ones in shape and type (N(0, 0.02) bf16 matrices), with
norm gammas around one. In whole models the embedding has std 0.1 and the two projections that
write the residual stream are small enough that a layer adds a part of the residual's size and not
several times it, as in trained decoders: the logits then have a clear winner, so that a whole
greedy generation can be compared.
"""

import math
import sys
from pathlib import Path

import numpy as np
import torch

sys.path.insert(0, str(Path(__file__).resolve().parent.parent / "llama1b-megakernel_amd"))

import mk_lib  # noqa: E402
from llama_with_megakernel import LlamaInferenceConfig, NeuronConfigLlamaMK, NeuronLlamaForCausalLM  # noqa: E402
from mk_config import LlamaDims  # noqa: E402
from mk_weights import pack_for_megakernel  # noqa: E402

LAYERS, HIDDEN, HEADS, KV_HEADS, HEAD_DIM, INTER, VOCAB = 16, 2048, 32, 8, 64, 8192, 128256
QKV = (HEADS + 2 * KV_HEADS) * HEAD_DIM
LAYER_PARAMS = QKV * HIDDEN + HIDDEN * HIDDEN + 3 * HIDDEN * INTER
EPS = 1e-5
CAP = 1024              # the sampler's most candidates
DEV = "cuda"


def listed():
    return [
        # one layer as its own launch, a 1024-row cache: the smallest call of the kernel seam
        {"name": "layer_b1_1k", "kind": "layer", "batch": 1, "rows": 1024, "lo": 1023, "hi": 1023},
        # a few sequences of short and unequal lengths
        {"name": "layer_b3_ragged", "kind": "layer", "batch": 3, "rows": 1000, "lo": 37, "hi": 901},
        # more than one 16-row tile of sequences, ragged, in a 4096-row cache
        {"name": "layer_b20_4k", "kind": "layer", "batch": 20, "rows": 4096, "lo": 211, "hi": 3999},
        # greedy generation at batch 1 behind a 384-token prompt, the benchmark's headline
        {"name": "loop_b1_32_steps", "kind": "loop", "steps": 32, "rows": 1024, "pos": 384},
        # whole steps: eight ragged conversations; 32 sequences near the end of 8192-row caches
        {"name": "step_b8_ragged", "kind": "step", "batch": 8, "rows": 4096, "lo": 539, "hi": 3179},
        {"name": "step_b32_8k", "kind": "step", "batch": 32, "rows": 8192, "lo": 8066, "hi": 8191},
        # time to the first token: the benchmark's prompt, and a long document
        {"name": "first_384", "kind": "first", "tokens": 384, "rows": 1024},
        {"name": "first_3001", "kind": "first", "tokens": 3001, "rows": 4096},
        # context encoding of one layer: a short turn late in a conversation, and a long prompt
        {"name": "prefill_33_at_700", "kind": "prefill", "tokens": 33, "start": 700, "rows": 1024},
        {"name": "prefill_1100", "kind": "prefill", "tokens": 1100, "start": 0, "rows": 2048},
        # sampling one sequence's next token (top-k 50, nucleus 0.9), and a batch of mixed settings
        {"name": "sample_b1", "kind": "sample", "batch": 1, "vocab": VOCAB, "mixed": False, "top_k": 50, "top_p": 0.9},
        {"name": "sample_b32_mixed", "kind": "sample", "batch": 32, "vocab": VOCAB, "mixed": True},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["layer", "layer", "step", "loop", "first", "prefill", "prefill", "sample"])
    if kind in ("layer", "step"):
        batch = 1 if rng.random() < 0.25 else rng.randint(2, 32)
        rows = _log_int(rng, 64, 8192)
        hi = rng.randint(rows // 2, rows - 1)
        lo = hi if batch == 1 else rng.randint(0, hi)
        return {"kind": kind, "batch": batch, "rows": rows, "lo": lo, "hi": hi}
    if kind == "loop":
        steps, pos = _log_int(rng, 1, 24), _log_int(rng, 1, 4000)
        return {"kind": kind, "steps": steps, "rows": pos + steps + rng.randint(0, 64), "pos": pos}
    if kind == "first":
        tokens = _log_int(rng, 2, 3001)
        return {"kind": kind, "tokens": tokens, "rows": tokens + rng.randint(0, 1000)}
    if kind == "prefill":
        tokens = _log_int(rng, 1, 4096)
        start = rng.choice([0, _log_int(rng, 1, 4000)])
        return {"kind": kind, "tokens": tokens, "start": start, "rows": tokens + start + rng.randint(0, 64)}
    vocab = VOCAB if rng.random() < 0.6 else _log_int(rng, 1000, VOCAB)
    case = {"kind": kind, "batch": rng.randint(1, 32), "vocab": vocab, "mixed": rng.random() < 0.4}
    if not case["mixed"]:
        case["top_k"], case["top_p"] = rng.choice([0, 1, rng.randint(2, CAP)]), round(rng.uniform(0.5, 1.0), 3)
    return case


# -- inputs ---------------------------------------------------------------------------------


def _gen(seed, what):
    return torch.Generator(device=DEV).manual_seed(seed * 1009 + what)


def _normal(shape, std, gen):
    return torch.empty(shape, dtype=torch.bfloat16, device=DEV).normal_(0.0, std, generator=gen)


def _state_dict(layers, seed):
    """Weights under the names of the checkpoint format, on the GPU."""
    g = _gen(seed, 1)
    out_std = 0.02 if layers == 1 else 0.005 / math.sqrt(2 * layers)
    sd = {"embed_tokens.weight": _normal((VOCAB, HIDDEN), 0.1, g)}
    for i in range(layers):
        p = "layers.%d." % i
        for name, shape, std in (("self_attn.q_proj", (HIDDEN, HIDDEN), 0.02),
                                 ("self_attn.k_proj", (KV_HEADS * HEAD_DIM, HIDDEN), 0.02),
                                 ("self_attn.v_proj", (KV_HEADS * HEAD_DIM, HIDDEN), 0.02),
                                 ("self_attn.o_proj", (HIDDEN, HIDDEN), out_std),
                                 ("mlp.gate_proj", (INTER, HIDDEN), 0.02),
                                 ("mlp.up_proj", (INTER, HIDDEN), 0.02),
                                 ("mlp.down_proj", (HIDDEN, INTER), out_std)):
            sd[p + name + ".weight"] = _normal(shape, std, g)
        for name in ("input_layernorm", "post_attention_layernorm"):
            sd[p + name + ".weight"] = _normal((HIDDEN,), 0.1, g) + 1
    sd["norm.weight"] = _normal((HIDDEN,), 0.1, g) + 1
    return sd


def _fill_cache(kv, seed):
    """Rows of earlier tokens: [layers, 2, batch, kv heads, rows, head dim]. The keys' size
    differs from head to head, so some heads look at few rows and some at many."""
    kv.normal_(0.0, 1.0, generator=_gen(seed, 2))
    kv[:, 0] *= torch.tensor([0.5, 1, 2, 1, 0.5, 1, 4, 1], dtype=torch.bfloat16, device=DEV).view(1, 1, KV_HEADS, 1, 1)
    return kv


def _positions(case, seed):
    b, lo, hi = case["batch"], case["lo"], case["hi"]
    pos = np.array([hi] if b == 1 else [lo + (hi - lo) * i // (b - 1) for i in range(b)], dtype=np.int32)
    return torch.from_numpy(np.random.RandomState(seed % (1 << 31)).permutation(pos)).to(DEV)


def _ids(n, seed):
    return torch.randint(0, VOCAB, (n,), generator=_gen(seed, 3), device=DEV, dtype=torch.int32)


def _hidden(n, seed):
    """A residual stream as the middle layers see it: a few channels are much larger."""
    g = _gen(seed, 4)
    h = torch.randn(n, HIDDEN, generator=g, device=DEV)
    h[:, torch.randint(0, HIDDEN, (8,), generator=g, device=DEV)] *= 10
    return h.to(torch.bfloat16)


def _sampling_inputs(case, seed):
    b, v = case["batch"], case["vocab"]
    logits = torch.randn(b, v, generator=_gen(seed, 5), device=DEV) * 2.5
    if not case["mixed"]:
        rows = [(case["top_k"], case["top_p"], 0.8)]
    else:
        rows = [(50, 0.9, 0.8), (1, 1.0, 1.0), (0, 0.95, 1.0), (40, 1.0, 0.7), (1000, 0.9, 1.2)]
    rows = [rows[i % len(rows)] for i in range(b)]
    counter = torch.randint(0, 8192, (b,), generator=_gen(seed, 6), device=DEV, dtype=torch.int32)
    return logits, rows, counter


def _model(rows, batch, seed):
    config = LlamaInferenceConfig(NeuronConfigLlamaMK(batch_size=batch, seq_len=rows, max_context_length=rows))
    model = NeuronLlamaForCausalLM("random:%d" % seed, config)
    model.packed = model.convert_hf_to_neuron_state_dict(_state_dict(LAYERS, seed), config, device=DEV)
    model.load()
    return model


def prepare(case, seed):
    kind = case["kind"]
    s = {"kind": kind}
    if kind == "sample":
        logits, rows, s["counter"] = _sampling_inputs(case, seed)
        s["logits"], s["seed"] = logits, seed
        s["params"] = mk_lib.prepare_sampling_params(len(rows), *(list(c) for c in zip(*rows)))
        s["tokens"] = torch.zeros(len(rows), dtype=torch.int32, device=DEV)
        s["uniforms"] = torch.zeros(len(rows), dtype=torch.float32, device=DEV)
    elif kind in ("layer", "prefill"):
        n = case["batch"] if kind == "layer" else 1
        packed = pack_for_megakernel(_state_dict(1, seed), LlamaDims(n_layers=1), device=DEV, rope_rows=case["rows"])
        s["packed"], s["weights"] = packed, mk_lib.weights_struct(packed)
        kv = torch.empty(1, 2, n, KV_HEADS, case["rows"], HEAD_DIM, dtype=torch.bfloat16, device=DEV)
        s["kv"] = _fill_cache(kv, seed)
        if kind == "layer":
            s["ws"] = mk_lib.Workspace(n, case["rows"], torch.device(DEV))
            s["pos"], s["hidden"], s["out"] = _positions(case, seed), _hidden(n, seed), torch.empty(
                n, HIDDEN, dtype=torch.bfloat16, device=DEV)
        else:
            s["ids"], s["start"] = _ids(case["tokens"], seed), case["start"]
            s["ws"] = mk_lib.prefill_workspace(min(case["tokens"], 4096), DEV)
            s["out"] = torch.empty(case["tokens"], HIDDEN, dtype=torch.bfloat16, device=DEV)
    else:
        m = s["model"] = _model(case["rows"], case.get("batch", 1), seed)
        if kind == "first":
            s["ids"] = _ids(case["tokens"], seed)
        else:
            _fill_cache(m.kv, seed)
            s["ids"] = _ids(case.get("batch", 1), seed)
            if kind == "step":
                s["pos"] = _positions(case, seed)
            else:
                s["pos"] = torch.full((1,), case["pos"], dtype=torch.int32, device=DEV)
                s["tokens"] = torch.zeros(case["steps"], dtype=torch.int32, device=DEV)
    return s


def run(s):
    kind = s["kind"]
    if kind == "sample":
        mk_lib.sample(s["logits"], s["params"], s["tokens"], seed=s["seed"], counter=s["counter"], uniforms_out=s["uniforms"])
        return {"tokens": s["tokens"], "uniforms": s["uniforms"]}
    if kind == "layer":
        k, v = s["kv"][0]
        mk_lib.decode_step(s["weights"], s["ws"], [k], [v], s["pos"], hidden_in=s["hidden"], hidden_out=s["out"],
                           batch=k.shape[0])
        return {"hidden": s["out"], "kv": s["kv"]}
    if kind == "prefill":
        k, v = s["kv"][0]
        mk_lib.prefill(s["weights"], s["ids"], [k], [v], s["start"], s["ws"], hidden_out=s["out"])
        return {"hidden": s["out"], "kv": s["kv"]}
    m = s["model"]
    if kind == "step":
        logits, _ = m.forward(input_ids=s["ids"], position_ids=s["pos"])
        return {"logits": logits, "tokens": m.tokens, "kv": m.kv}
    if kind == "loop":
        mk_lib.decode_loop(m.weights, m.ws, m.k_caches, m.v_caches, s["pos"], s["ids"], s["tokens"].numel(),
                           tokens_out=s["tokens"], logits=m.logits, hidden_out=m.hidden_out)
        return {"logits": m.logits, "tokens": s["tokens"], "hidden": m.hidden_out, "kv": m.kv}
    m.prefill(s["ids"])
    m.launcher("decode").launch()
    return {"logits": m.logits, "tokens": m.tokens, "hidden": m.hidden_out, "kv": m.kv}


# -- what a pass cannot do without -------------------------------------------------------------


def work(case):
    kind = case["kind"]
    row = KV_HEADS * HEAD_DIM * 2 * 2           # a K and a V row of one layer, bytes
    if kind == "sample":
        n = case["batch"] * case["vocab"]
        return {"bytes": 4 * n + 24 * case["batch"], "flops": 2 * n}
    head_bytes, head_flops = VOCAB * HIDDEN * 2, 2 * VOCAB * HIDDEN
    if kind in ("layer", "step"):
        b, lo, hi = case["batch"], case["lo"], case["hi"]
        seen = hi if b == 1 else sum(lo + (hi - lo) * i // (b - 1) for i in range(b))
        layers = 1 if kind == "layer" else LAYERS
        byt = layers * (LAYER_PARAMS * 2 + row * (seen + b)) + 4 * b * HIDDEN
        flops = layers * (2 * b * LAYER_PARAMS + 4 * HIDDEN * (seen + b))
        if kind == "step":
            byt, flops = byt + head_bytes + 4 * b * VOCAB, flops + b * head_flops
        return {"bytes": byt, "flops": flops}
    if kind == "loop":                          # the weights once for each step: a step needs the last one's token
        n, p = case["steps"], case["pos"]
        seen = sum(range(p, p + n))
        return {"bytes": n * (LAYERS * LAYER_PARAMS * 2 + head_bytes) + LAYERS * row * (seen + n) + 4 * VOCAB,
                "flops": n * (2 * LAYERS * LAYER_PARAMS + head_flops) + 4 * LAYERS * HIDDEN * (seen + n)}
    n, start = case["tokens"], case.get("start", 0)
    pairs = n * start + n * (n + 1) // 2        # (token, row it looks at)
    if kind == "prefill":
        return {"bytes": LAYER_PARAMS * 2 + row * (start + n) + 4 * n * HIDDEN,
                "flops": 2 * n * LAYER_PARAMS + 4 * HIDDEN * pairs}
    # the last layer needs only the keys and values of all tokens but the last
    kv_params = 2 * KV_HEADS * HEAD_DIM * HIDDEN
    return {"bytes": LAYERS * LAYER_PARAMS * 2 + LAYERS * row * n + n * HIDDEN * 2 + head_bytes + 4 * VOCAB,
            "flops": (LAYERS - 1) * (2 * n * LAYER_PARAMS + 4 * HIDDEN * pairs) + 2 * n * kv_params
            + 2 * LAYER_PARAMS + 4 * HIDDEN * n + head_flops}


def tolerance(case):
    kind = case["kind"]
    if kind == "sample":
        return "exact"
    # About four times the error against 64 bits that one layer shows (0.0035 for a decode step; 0.006 to
    # 0.0095 for context encoding, which also rounds the attention's weights to bf16 and starts from the
    # small embedding), and twice that of 16 layers in a row (0.014).
    if kind in ("layer", "prefill"):
        return {"rel": 1.2e-2 if kind == "layer" else 2.5e-2, "max": 0.15}
    return {"rel": 2.8e-2, "max": 0.3, "differ": 0.0}


# -- the same in 64 bits, as plain torch ----------------------------------------------------------


def _rope(pos):
    """cos and sin for each position, [n, head dim] each: bf16 by the model's definition."""
    base = 500000.0 ** (-np.arange(0, HEAD_DIM, 2) / HEAD_DIM)
    wl = 2 * np.pi / base
    smooth = (8192 / wl - 1) / 3
    mid = (1 - smooth) * base / 8 + smooth * base
    inv = np.where(wl < 2048, base, np.where(wl > 8192, base / 8, mid)).astype(np.float32)
    f = pos.double()[:, None] * torch.from_numpy(np.concatenate([inv, inv])).to(DEV).double()[None]
    return f.cos().bfloat16().double(), f.sin().bfloat16().double()


def _rotate(x, cos, sin):
    """x: [n, heads, head dim]."""
    a, b = x.chunk(2, -1)
    return x * cos[:, None] + torch.cat([-b, a], -1) * sin[:, None]


def _norm(x):
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS)


def _exact_layer(sd, i, h, pos, kv, owner):
    """One decoder layer for tokens h [n, hidden] at rows pos [n] of sequences owner (one of each sequence,
    or consecutive tokens of sequence 0). kv: [2, batch, kv heads, rows, head dim], written in place."""
    def w(name, gamma=None):
        t = sd["layers.%d.%s.weight" % (i, name)]
        if gamma is not None:                   # folded at load time, in 32 bits, and kept in bf16
            t = (t.float() * sd["layers.%d.%s.weight" % (i, gamma)].float()).bfloat16()
        return t.double().t()

    n = h.shape[0]
    x, (cos, sin) = _norm(h), _rope(pos)
    q = _rotate((x @ w("self_attn.q_proj", "input_layernorm")).view(n, HEADS, HEAD_DIM), cos, sin)
    k = _rotate((x @ w("self_attn.k_proj", "input_layernorm")).view(n, KV_HEADS, HEAD_DIM), cos, sin)
    v = (x @ w("self_attn.v_proj", "input_layernorm")).view(n, KV_HEADS, HEAD_DIM)
    at, idx = pos.long(), owner.long()
    kv[0][idx, :, at], kv[1][idx, :, at] = k, v
    out = torch.empty(n, HEADS, HEAD_DIM, dtype=torch.float64, device=DEV)
    grouped = q.view(n, KV_HEADS, HEADS // KV_HEADS, HEAD_DIM)
    for b in idx.unique().tolist():
        rows = (idx == b).nonzero()[:, 0]
        last = at[rows].max().item() + 1
        mask = torch.arange(last, device=DEV)[None] > at[rows][:, None]
        for g in range(KV_HEADS):
            keys, vals = kv[0, b, g, :last].double(), kv[1, b, g, :last].double()
            qs = grouped[rows, g].reshape(-1, HEAD_DIM)
            sc = (qs @ keys.t().contiguous() / math.sqrt(HEAD_DIM)).view(len(rows), -1, last)
            p = sc.masked_fill(mask[:, None], float("-inf")).softmax(-1)
            out[rows, g * (HEADS // KV_HEADS):(g + 1) * (HEADS // KV_HEADS)] = (p.view(-1, last) @ vals).view(
                len(rows), -1, HEAD_DIM)
    h = h + out.view(n, HIDDEN) @ w("self_attn.o_proj")
    x = _norm(h)
    gate = x @ w("mlp.gate_proj", "post_attention_layernorm")
    act = gate * torch.sigmoid(gate) * (x @ w("mlp.up_proj", "post_attention_layernorm"))
    return h + act @ w("mlp.down_proj")


def _exact_head(sd, h):
    x = _norm(h) * sd["norm.weight"].double()
    return torch.cat([x @ c.double().t() for c in sd["embed_tokens.weight"].chunk(8)], -1)


def _philox(counter, row, seed):
    """First word of Philox4x32-10."""
    c, k = [counter, row, 0, 0], [seed & 0xFFFFFFFF, seed >> 32 & 0xFFFFFFFF]
    for _ in range(10):
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [p1 >> 32 ^ c[1] ^ k[0], p1 & 0xFFFFFFFF, p0 >> 32 ^ c[3] ^ k[1], p0 & 0xFFFFFFFF]
        k = [k[0] + 0x9E3779B9 & 0xFFFFFFFF, k[1] + 0xBB67AE85 & 0xFFFFFFFF]
    return c[0]


def _exact_sample(case, seed):
    logits, rows, counter = _sampling_inputs(case, seed)
    tokens, uniforms = [], []
    for b, (top_k, top_p, temp) in enumerate(rows):
        if top_k == 1:
            tokens.append(int(logits[b].argmax()))
            uniforms.append(-1.0)
            continue
        u = (_philox(int(counter[b]), b, seed) >> 8) / 2.0 ** 24
        x, at = logits[b].double().sort(descending=True, stable=True)
        k = min(top_k if 0 < top_k <= CAP else CAP, x.numel())
        n = int((x >= x[k - 1]).sum())
        cum = ((x[:n] - x[0]) / temp).exp().cumsum(0)
        before = cum - ((x[:n] - x[0]) / temp).exp()
        keep = int((before < top_p * cum[-1]).sum()) if 0 < top_p < 1 else n
        pick = min(int((cum[:keep] <= u * cum[keep - 1]).sum()), keep - 1)
        tokens.append(int(at[pick]))
        uniforms.append(u)
    return {"tokens": torch.tensor(tokens, dtype=torch.int32), "uniforms": torch.tensor(uniforms, dtype=torch.float64)}


def exact(case, seed):
    kind = case["kind"]
    if kind == "sample":
        return _exact_sample(case, seed)
    if kind in ("layer", "prefill"):
        sd = _state_dict(1, seed)
        batch = case["batch"] if kind == "layer" else 1
        kv = _fill_cache(torch.empty(1, 2, batch, KV_HEADS, case["rows"], HEAD_DIM, dtype=torch.bfloat16, device=DEV), seed)
        kv = kv.double()
        if kind == "layer":
            h, pos, owner = _hidden(batch, seed).double(), _positions(case, seed), torch.arange(batch, device=DEV)
        else:
            h = sd["embed_tokens.weight"][_ids(case["tokens"], seed).long()].double()
            pos = torch.arange(case["start"], case["start"] + case["tokens"], device=DEV)
            owner = torch.zeros_like(pos)
        return {"hidden": _exact_layer(sd, 0, h, pos, kv[0], owner), "kv": kv}
    sd, embed = _state_dict(LAYERS, seed), None
    embed = sd["embed_tokens.weight"]
    batch = case.get("batch", 1)
    kv = torch.zeros(LAYERS, 2, batch, KV_HEADS, case["rows"], HEAD_DIM, dtype=torch.bfloat16, device=DEV)
    if kind != "first":
        _fill_cache(kv, seed)
    big = kv.numel() > 1 << 30                  # its copy in 64 bits would take tens of GB: a layer's at a time, none returned
    if not big:
        kv = kv.double()

    def forward(ids, pos, owner):
        h = embed[ids.long()].double()
        for i in range(LAYERS):
            h = _exact_layer(sd, i, h, pos, kv[i].double() if big else kv[i], owner)
        return h

    if kind == "loop":
        tok, got = _ids(1, seed), []
        for t in range(case["steps"]):
            pos = torch.full((1,), case["pos"] + t, device=DEV)
            h = forward(tok, pos, torch.zeros_like(pos))
            logits = _exact_head(sd, h)
            tok = logits.argmax(-1)
            got.append(tok)
        return {"logits": logits, "tokens": torch.cat(got).int(), "hidden": h, "kv": kv}
    if kind == "step":
        pos = _positions(case, seed)
        logits = _exact_head(sd, forward(_ids(batch, seed), pos, torch.arange(batch, device=DEV)))
        return {"logits": logits, "tokens": logits.argmax(-1).int(), "kv": None if big else kv}
    pos = torch.arange(case["tokens"], device=DEV)
    h = forward(_ids(case["tokens"], seed), pos, torch.zeros_like(pos))[-1:]
    logits = _exact_head(sd, h)
    return {"logits": logits, "tokens": logits.argmax(-1).int(), "hidden": h, "kv": kv}
