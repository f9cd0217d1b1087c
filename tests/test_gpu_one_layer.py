"""The batched kernel's one-layer instantiations (``mk_batch_one.hip``) against
its looping ones: two one-layer steps, the second on the first's hidden state,
give the bits of one two-layer step — hidden state, K/V rows, logits and greedy
tokens — at batches on both sides of the 16-token tile, from token ids and from
hidden states, at ragged positions that reach every split of the attention.
"""

import pytest
import torch

from gpu_common import need_gpu, packed_on_device

pytestmark = pytest.mark.gpu

S = 1500


@pytest.fixture(scope="module")
def packed():
    need_gpu()
    from mk_config import LlamaDims
    from mk_weights import param_specs
    d = LlamaDims(n_layers=2)
    g = torch.Generator(device="cuda").manual_seed(9)
    sd = {n: torch.ones(s, dtype=torch.bfloat16, device="cuda") if kind == "ones" else
          torch.empty(s, dtype=torch.bfloat16, device="cuda").normal_(0, 0.02, generator=g)
          for n, s, kind in param_specs(d)}
    return packed_on_device(sd, d, S)


@pytest.mark.parametrize("from_tokens", [True, False])
@pytest.mark.parametrize("batch", [2, 8, 9, 16, 17, 32])
def test_one_layer_steps_equal_the_loop(packed, batch, from_tokens):
    import mk_lib
    w = mk_lib.weights_struct(packed)
    g = torch.Generator(device="cuda").manual_seed(batch)
    kv = torch.empty(2, 2, batch, 8, S, 64, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    pos = torch.tensor([(S - 1) * b // (batch - 1) for b in range(batch)], dtype=torch.int32, device="cuda")
    ids = torch.randint(0, 128256, (batch,), generator=g, device="cuda", dtype=torch.int32)
    x = torch.empty(batch, 2048, dtype=torch.bfloat16, device="cuda").normal_(generator=g)
    ws = mk_lib.Workspace(batch, S, torch.device("cuda"))
    first = dict(tokens=ids) if from_tokens else dict(hidden_in=x)

    def outputs():
        return (torch.zeros(batch, 2048, dtype=torch.bfloat16, device="cuda"),
                torch.zeros(batch, 128256, device="cuda"), torch.zeros(batch, dtype=torch.int32, device="cuda"))

    kv2 = kv.clone()
    hid, logits, tok = outputs()
    mk_lib.decode_step(w, ws, list(kv2[:, 0]), list(kv2[:, 1]), pos, hidden_out=hid, logits=logits, next_token=tok,
                       batch=batch, **first)
    kv1 = kv.clone()
    mid, hid1, (_, logits1, tok1) = torch.zeros_like(hid), torch.zeros_like(hid), outputs()
    mk_lib.decode_step(w, ws, [kv1[0, 0]], [kv1[0, 1]], pos, hidden_out=mid, batch=batch, **first)
    mk_lib.decode_step(w, ws, [kv1[1, 0]], [kv1[1, 1]], pos, hidden_in=mid, hidden_out=hid1, logits=logits1,
                       next_token=tok1, first_layer=1, batch=batch)
    torch.cuda.synchronize()
    assert ws.read_device_error() == 0
    assert torch.equal(hid.view(torch.int16), hid1.view(torch.int16))
    assert torch.equal(kv2.view(torch.int16), kv1.view(torch.int16))
    assert torch.equal(logits.view(torch.int32), logits1.view(torch.int32)) and torch.equal(tok, tok1)
