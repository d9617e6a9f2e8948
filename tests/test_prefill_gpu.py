"""The prompt passes of OlmoDecoder.prefill against the one-token step at every position: caches, logits, next token and
position equal bit for bit, for each weight kind, for prompts on both sides of the launches' row limits (a pass of one
row, 16 and 17 rows, two and three passes of 32; at the shipped pass of 256 rows 65, 160, 256 and 257 tokens), with whole
and with split plans of the linears, and over a cache that an earlier, longer prompt has filled."""

from __future__ import annotations

import pytest
import torch

from byteprof_amd.optim import olmo as OG
from byteprof_amd.optim import skinny as S

pytestmark = pytest.mark.gpu

DEV = torch.device("cuda:0")
CFGS = {"fused": OG.OlmoConfig(hidden=1024, ffn=1024, layers=2, heads=8, vocab=512, max_len=96),
        "odd": OG.OlmoConfig(hidden=384, ffn=640, layers=3, heads=6, vocab=1000, max_len=96)}


def _check_prompts(dec, lengths, seed=1):
    cfg = dec.cfg
    g = torch.Generator().manual_seed(seed)
    for length in lengths:
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


@pytest.mark.parametrize("kind", ["bf16", "int8", "int4"])
@pytest.mark.parametrize("shape", ["fused", "odd"])
def test_prefill_equals_the_one_token_steps(kind, shape, monkeypatch):
    cfg = CFGS[shape]
    dec = OG.OlmoDecoder(cfg, OG.random_weights(cfg, DEV, seed=5), kind)
    monkeypatch.setattr(OG, "PREFILL_ROWS", 32)
    _check_prompts(dec, (90, 1, 2, 16, 17, 33, 64, 65))


@pytest.mark.parametrize("kind", ["bf16", "int8", "int4"])
def test_prefill_at_its_own_pass_size(kind):
    """Passes of PREFILL_ROWS rows: the launches past 64 rows, one full pass, and a second pass of one row."""
    cfg = OG.OlmoConfig(hidden=384, ffn=640, layers=2, heads=6, vocab=1000, max_len=288)
    assert OG.PREFILL_ROWS == 256
    dec = OG.OlmoDecoder(cfg, OG.random_weights(cfg, DEV, seed=6), kind)
    _check_prompts(dec, (257, 65, 160, 256))


def _split_two(monkeypatch):
    """Every plan outside a user cfg with K split two ways."""
    table, int4 = S._table_plan, S.int4_cfg
    monkeypatch.setattr(S, "_table_plan", lambda *a, **k: (*table(*a, **k)[:2], 2, 0))
    monkeypatch.setattr(S, "int4_cfg", lambda n, k, tile, cfg=None: int4(n, k, tile, cfg) if cfg is not None else
                        (int4(n, k, tile)[0], 2))
    S._own_plan.cache_clear()


@pytest.fixture
def split_plans(monkeypatch):
    _split_two(monkeypatch)
    yield
    S._own_plan.cache_clear()


@pytest.mark.parametrize("kind", ["bf16", "int8", "int4"])
def test_split_plans_of_every_linear(kind, split_plans, monkeypatch):
    """A decoder whose plans all split K (no norm prologue, no SiLU epilogue, the down projection's partials reduced with the
    norm in verify passes): prompts against steps, steps and verify passes against the same decoder without splits within the
    rounding of the sums, and the branches taken."""
    cfg = CFGS["fused"]
    weights = OG.random_weights(cfg, DEV, seed=7)
    dec = OG.OlmoDecoder(cfg, weights, kind)
    H, F, V = cfg.hidden, cfg.ffn, cfg.vocab
    assert all(dec._plan(n, k, r)[2] == 2 for n, k in ((3 * H, H), (H, H), (2 * F, H), (H, F), (V, H)) for r in (1, 9))
    assert not dec.fuse_norms and (dec._down_splitk(9) is not None) == (kind != "int4")
    monkeypatch.setattr(OG, "PREFILL_ROWS", 32)
    _check_prompts(dec, (90, 2, 17, 33))
    assert "gu" in dec._prefill and dec._prefill["ws"].numel() >= 2 * 32 * 3 * H
    prompt = torch.randint(0, V, (40,), generator=torch.Generator().manual_seed(3))
    dec.prefill(prompt)
    logits = dec.logits.clone()
    steps = []
    dec.pos.zero_()
    for t in prompt.tolist():
        dec.tok.fill_(t)
        dec.step()
        steps.append(dec.logits.clone())
    dec.verify_buffers(16)
    for s in (1, 3, 9, 16):
        dec.v_ids[:s].copy_(prompt[-s:])
        dec.v_pos.fill_(len(prompt) - s)
        dec.verify(s)
        assert torch.equal(dec.vlogits[:s], torch.cat(steps[-s:])), s
    monkeypatch.undo()
    S._own_plan.cache_clear()
    whole = OG.OlmoDecoder(cfg, weights, kind)
    whole.prefill(prompt)
    diff = (whole.logits.float() - logits.float()).norm() / whole.logits.float().norm()
    assert 0 < diff < 2e-2  # two sums of K / 2 instead of one, through two layers of bf16 roundings (2^-8 each)


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
