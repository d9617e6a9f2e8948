"""The prompt passes of OlmoDecoder.prefill against the one-token step at every position: caches, logits, next token and
position equal bit for bit, for each weight kind, for prompts on both sides of the launches' row limits (a pass of one
row, 16 and 17 rows, two and three passes), with fused and with split plans, and over a cache that an earlier, longer
prompt has filled."""

from __future__ import annotations

import pytest
import torch

from byteprof_amd.optim import olmo as OG

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
CFGS = {"fused": OG.OlmoConfig(hidden=1024, ffn=1024, layers=2, heads=8, vocab=512, max_len=96),
        "odd": OG.OlmoConfig(hidden=384, ffn=640, layers=3, heads=6, vocab=1000, max_len=96)}


@pytest.mark.parametrize("kind", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("shape", ["fused", "odd"])
def test_prefill_equals_the_one_token_steps(kind, shape, monkeypatch):
    cfg = CFGS[shape]
    dec = OG.OlmoDecoder(cfg, OG.random_weights(cfg, DEV, seed=5), kind)
    monkeypatch.setattr(OG, "PREFILL_ROWS", 32)
    g = torch.Generator().manual_seed(1)
    for length in (90, 1, 2, 16, 17, 33, 64, 65):
        ids = torch.randint(0, cfg.vocab, (length,), generator=g)
        dec.prefill(ids)
        got = [t.clone() for t in (dec.k_cache[:, :, :length], dec.v_cache[:, :, :length], dec.logits, dec.tok, dec.pos)]
        dec.pos.zero_()
        for t in ids.tolist():
            dec.tok.fill_(t)
            dec.step()
        want = (dec.k_cache[:, :, :length], dec.v_cache[:, :, :length], dec.logits, dec.tok, dec.pos)
        for name, a, b in zip(("k", "v", "logits", "tok", "pos"), got, want):
            assert torch.equal(a, b), (length, name)
        assert torch.isfinite(dec.logits.float()).all() and int(dec.pos) == length


def test_prompts_inside_and_outside_inference_mode():
    """The pass buffers are made at the first prompt: one inside torch.inference_mode, then one outside it, and a
    generate() each way, give the same tokens."""
    cfg = CFGS["odd"]
    dec = OG.OlmoDecoder(cfg, OG.random_weights(cfg, DEV, seed=5), "bf16")
    gen = OG.make_generate(dec)
    prompt = torch.tensor([[5, 9, 2, 700, 31]])
    with torch.inference_mode():
        inside = gen(prompt, max_new_tokens=4)
    outside = gen(prompt, max_new_tokens=4)
    assert torch.equal(inside.cpu(), outside.cpu())
