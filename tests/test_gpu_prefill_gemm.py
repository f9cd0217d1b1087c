"""GPU parity of one prefill layer (``mk_prefill`` with the hidden state out)
at row counts around the edges of its GEMM tiles and K splits, and behind
caches long enough for its attention to split the keys.

The projections run on output tiles from 64x64 to 256x256, with K split into
partials for few tokens, chosen by row count; the counts here lie on both
sides of the tiles' and the splits' edges and reach every tile of every
projection, on rows that are and that are not a multiple of 16. The attention
takes 16 or 32 tokens per workgroup in steps of 64 keys and, for few tokens
behind many rows, splits the keys over workgroups. For each count and start:

* the hidden state and the K/V rows against plain torch on the GPU: fp32
  products with bf16 rounding at the kernel's points ("rounded") and float64
  without any ("exact"). The kernel's departure from exact may be at most 1.5
  times the rounded reference's (rms), the bound of the decode layer tests: it
  rounds at the same points and differs in the order of fp32 sums, and in the
  attention's weights, rounded to bf16 relative to a running maximum;
* the row-major weights give the same bits as their MFMA-tiled copies;
* rows outside the prompt keep their bytes.
"""

import math

import pytest
import torch

from gpu_common import need_gpu, say

pytestmark = pytest.mark.gpu

S, START = 4200, 5
LATE = [(64, 64), (123, 5), (124, 5), (128, 0), (128, 1), (1, 600), (1, 4199), (16, 3000), (33, 700), (65, 1983), (128, 2900), (129, 4031), (384, 2690), (500, 3700)]
COUNTS = [1, 16, 17, 63, 64, 65, 127, 128, 129, 192, 257, 384, 385, 513, 641, 700, 900, 1025, 1281, 1600, 2049, 3001, 3100, 3400, 4077]


@pytest.fixture(scope="module")
def layer():
    need_gpu()
    import mk_lib
    from mk_config import LlamaDims
    from mk_weights import pack_for_megakernel, param_specs
    d = LlamaDims(n_layers=1)
    g = torch.Generator(device="cuda").manual_seed(3)
    sd = {n: torch.ones(s, dtype=torch.bfloat16, device="cuda") if kind == "ones" else
          torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(0, 0.02, generator=g)
          for n, s, kind in param_specs(d)}
    packed = pack_for_megakernel(sd, d, device="cuda", rope_rows=S)
    ids = torch.randint(0, d.vocab, (max(COUNTS),), generator=g, device="cuda", dtype=torch.int32)
    kv = torch.empty(2, 8, S, 64, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    return {"sd": sd, "packed": packed, "tiled": mk_lib.weights_struct(packed),
            "rows": mk_lib.weights_struct(packed, tiled=False), "ids": ids, "kv": kv}


def reference(layer, n, start, dt):
    """Hidden state, K and V rows of n tokens at row start: bf16 rounding at the
    kernel's points for dt float32, none for float64."""
    r = (lambda t: t.bfloat16().to(dt)) if dt == torch.float32 else (lambda t: t)
    sd, rope = layer["sd"], layer["packed"]["rope"][start:start + n].to(dt)
    w = lambda name: sd["layers.0." + name + ".weight"].to(dt).t()
    norm = lambda t: r(t * torch.rsqrt(t.square().mean(-1, keepdim=True) + 1e-5))

    def rot(t):
        a, b = t.chunk(2, -1)
        c, s = rope[:, None, :64], rope[:, None, 64:]
        return r(r(t * c) + r(torch.cat([-b, a], -1) * s))

    h = sd["embed_tokens.weight"][layer["ids"][:n].long()].to(dt)
    x = norm(h)
    q = rot(r(x @ w("self_attn.q_proj")).view(n, 32, 64))
    k = rot(r(x @ w("self_attn.k_proj")).view(n, 8, 64))
    v = r(x @ w("self_attn.v_proj")).view(n, 8, 64)
    keys = torch.cat([layer["kv"][0, :, :start].to(dt), k.transpose(0, 1)], 1)      # [8, start + n, 64]
    vals = torch.cat([layer["kv"][1, :, :start].to(dt), v.transpose(0, 1)], 1)
    mask = torch.arange(start + n, device="cuda")[None] > start + torch.arange(n, device="cuda")[:, None]
    att = torch.empty(n, 32, 64, dtype=dt, device="cuda")
    for hd in range(32):
        s = (q[:, hd] @ keys[hd // 4].t().contiguous() / math.sqrt(64)).masked_fill(mask, float("-inf"))
        p = torch.exp(s - s.amax(-1, keepdim=True))
        att[:, hd] = (r(p) @ vals[hd // 4]) / p.sum(-1, keepdim=True)
    h1 = r(h + r(r(att).view(n, 2048) @ w("self_attn.o_proj")))
    x = norm(h1)
    gate = x @ w("mlp.gate_proj")
    act = r(gate * torch.sigmoid(gate) * (x @ w("mlp.up_proj")))
    return r(h1 + r(act @ w("mlp.down_proj"))), k, v


def run(layer, n, start, weights):
    import mk_lib
    kv = layer["kv"].clone()
    out = torch.empty(n, 2048, dtype=torch.bfloat16, device="cuda")
    mk_lib.prefill(weights, layer["ids"][:n].contiguous(), [kv[0]], [kv[1]], start, mk_lib.prefill_workspace(n, "cuda"),
                   hidden_out=out)
    torch.cuda.synchronize()
    return out, kv


@pytest.mark.parametrize("n,start", [(n, START) for n in COUNTS] + LATE)
def test_layer_at_row_count(layer, n, start):
    out, kv = run(layer, n, start, layer["tiled"])
    again, kv2 = run(layer, n, start, layer["rows"])
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))
    assert torch.equal(kv.view(torch.int16), kv2.view(torch.int16))
    rounded, exact = reference(layer, n, start, torch.float32), reference(layer, n, start, torch.float64)
    rows = slice(start, start + n)
    got = (out, kv[0, :, rows].transpose(0, 1), kv[1, :, rows].transpose(0, 1))
    rms = lambda t: t.double().square().mean().sqrt().item()
    ratios = [rms(g.double() - e) / rms(f.double() - e) for g, f, e in zip(got, rounded, exact)]
    say(f"[prefill gemm] {n} tokens at {start}: departure from exact over the rounded reference's: "
        + ", ".join(f"{x:.3f}" for x in ratios))
    assert max(ratios) <= 1.5, ratios
    rest = torch.ones(S, dtype=torch.bool, device="cuda")
    rest[rows] = False
    assert torch.equal(kv[:, :, rest].view(torch.int16), layer["kv"][:, :, rest].view(torch.int16))


@pytest.mark.parametrize("cut,n", [(cut, n) for cut in (1, 32, 63, 64) for n in (2, 33, 64, 65, 128) if cut < n])
def test_prompt_within_128_rows_in_any_chunks(layer, n, cut):
    """Whole or cut in two, a prompt within the first 128 rows gives the same
    bits."""
    import mk_lib
    out, kv = run(layer, n, 0, layer["tiled"])
    kv2 = layer["kv"].clone()
    out2 = torch.empty_like(out)
    ws = mk_lib.prefill_workspace(n, "cuda")
    for a, b in ((0, cut), (cut, n)):
        mk_lib.prefill(layer["tiled"], layer["ids"][a:b].clone(), [kv2[0]], [kv2[1]], a, ws, hidden_out=out2[a:b])
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), out2.view(torch.int16))
    assert torch.equal(kv.view(torch.int16), kv2.view(torch.int16))


@pytest.mark.parametrize("start", [1, 100, 250, 620, 700, 1999, 3000, 4070])
def test_short_turn_in_any_pieces(layer, start):
    """A turn of up to 128 tokens, cut into any smaller calls, gives the same bits
    at any row: the order of all of a token's sums follows from its row alone. The
    starts put the turn across row 128, where that order changes, across rows where
    the split of the keys changes (640, 2048, 3072, 4096) and across none, on and off
    the 16-row blocks."""
    import mk_lib
    n = 128
    out, kv = run(layer, n, start, layer["tiled"])
    ws = mk_lib.prefill_workspace(n, "cuda")
    for cuts in ((64,), (1, 2, 19, 33, 90), tuple(range(7, n, 7))):
        kv2 = layer["kv"].clone()
        out2 = torch.empty_like(out)
        for a, b in zip((0,) + cuts, cuts + (n,)):
            mk_lib.prefill(layer["tiled"], layer["ids"][a:b].clone(), [kv2[0]], [kv2[1]], start + a, ws,
                           hidden_out=out2[a:b])
        torch.cuda.synchronize()
        assert torch.equal(out.view(torch.int16), out2.view(torch.int16)), cuts
        assert torch.equal(kv.view(torch.int16), kv2.view(torch.int16)), cuts
