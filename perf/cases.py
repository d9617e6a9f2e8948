"""Workloads of the decode hot path, through the entry points a program calls: single linears, the linears of a
decoder block, the attention launch, the mLSTM drafting paths and whole decoder calls.

A case names its path and sizes; `prepare` makes what a program has in hand before the call (inputs, weights in their
stored format, a captured graph where the decode loops capture one), `run` makes one pass, `exact` restates the pass
in float64 torch. The paths:

  linear     one SkinnyLinear / Int8Linear call, eager: a layer swapped into a model that is not graph-captured
  linears    the seven linears of `layers` decoder blocks (q, k, v, o, gate, up, down), each SkinnyLinear on the input
             of its role, in one captured graph: the decode loops' use of the linears (1 row: a decode step; 2..17:
             verify rounds of a token model; up to 64: drafted bytes, short prompts)
  attention  q/k norm + RoPE + cache write + attention of `layers` layers over their caches, in one captured graph
  round      a fused mLSTM verify round of `layers` layers in one captured graph: multistep_fw over T drafted
             positions, accept, then lazy_commit of the accepted prefix
  steps      the per-step mLSTM verify path of one layer in one captured graph: mlstm_step_into per position into
             history slots, then commit_state of the accepted slot
  step       one OlmoDecoder decode step (captured) at a given position
  verify     one OlmoDecoder verify pass of `rows` rows (captured) at a given position
  prompt     generate(prompt, max_new_tokens=1): the time to the first token
"""

from __future__ import annotations

import math

import torch
import torch.nn as nn

from byteprof_amd import _lib
from byteprof_amd.optim import draft_core, draft_fused, olmo
from byteprof_amd.optim.skinny_linear import SkinnyLinear
from byteprof_amd.quant.integrate import Int8Linear

DEV = "cuda"
EPS = 1e-6
BF = torch.bfloat16
DTYPES = {"bf16": torch.bfloat16, "fp16": torch.float16, "fp32": torch.float32}
ROLES = (("q", "h", "h"), ("k", "h", "h"), ("v", "h", "h"), ("o", "h", "h"), ("gate", "f", "h"), ("up", "f", "h"),
         ("down", "h", "f"))  # name, outputs, inputs


def listed() -> list[dict]:
    return [
        # the smallest call: one 2048 x 2048 projection of a decode step, called from an uncaptured model
        {"name": "linear bf16 1 row", "path": "linear", "kind": "bf16", "n": 2048, "k": 2048, "rows": 1, "bias": False},
        # a layer whose sizes are no multiple of anything (the int8 tests' 1025 x 2049), a few drafted rows
        {"name": "linear int8 ragged", "path": "linear", "kind": "int8", "n": 1025, "k": 2049, "rows": 5, "bias": True},
        # the LM head at the widest launch (64 rows: the widest verify pass, the tail of a prompt)
        {"name": "head bf16 64 rows", "path": "linear", "kind": "bf16", "n": 100352, "k": 2048, "rows": 64,
         "bias": False},
        # verify rounds: 8 drafts + 1 on int8 weights; 32 drafted bytes + 1 on bf16; 19 + 1 on int4
        {"name": "linears int8 9 rows", "path": "linears", "kind": "int8", "hidden": 2048, "ffn": 8192, "layers": 4,
         "rows": 9},
        {"name": "linears bf16 33 rows", "path": "linears", "kind": "bf16", "hidden": 2048, "ffn": 8192, "layers": 4,
         "rows": 33},
        {"name": "linears int4 20 rows", "path": "linears", "kind": "int4", "hidden": 2048, "ffn": 8192, "layers": 4,
         "rows": 20},
        # one token at the end of a long context: the cache stream of 16 heads of 128
        {"name": "attention 1 row long", "path": "attention", "heads": 16, "head_dim": 128, "layers": 8, "rows": 1,
         "pos": 1900, "max_len": 2048},
        # byte drafting: 32 drafts + 1 through five mLSTM layers of 16 heads, 20 accepted
        {"name": "mlstm round", "path": "round", "dtype": "bf16", "nh": 16, "dq": 64, "dv": 128, "layers": 5, "t": 33,
         "accepted": 20},
        # the per-step path at four 256-wide heads, 16 positions, float32 inputs
        {"name": "mlstm steps", "path": "steps", "dtype": "fp32", "nh": 4, "dq": 256, "dv": 256, "t": 16, "accepted": 9},
        # the headline: one decode step of the 1B shape, bf16
        {"name": "decode step bf16", "path": "step", "kind": "bf16", "hidden": 2048, "ffn": 8192, "heads": 16,
         "layers": 16, "vocab": 100352, "pos": 300},
        # a verify round of 8 drafts + 1 on the int8 model
        {"name": "verify int8 9 rows", "path": "verify", "kind": "int8", "hidden": 2048, "ffn": 8192, "heads": 16,
         "layers": 16, "vocab": 100352, "pos": 700, "rows": 9},
        # a prompt of a short paragraph up to its first token
        {"name": "prompt bf16 160", "path": "prompt", "kind": "bf16", "hidden": 2048, "ffn": 8192, "heads": 16,
         "layers": 16, "vocab": 100352, "tokens": 160},
    ]


def _log(rng, lo: int, hi: int) -> int:
    return min(hi, max(lo, round(math.exp(rng.uniform(math.log(lo), math.log(hi))))))


def draw(rng) -> dict:
    """One more case: the paths in about the listed proportions, sizes over the ranges the listed cases stand for."""
    path = rng.choice(["linear", "linear", "linear", "linears", "linears", "linears", "attention", "round", "steps",
                       "model"])
    kind = rng.choice(["bf16", "int8", "int4"])
    if path == "linear":
        n, k, rows = _log(rng, 64, 16384), _log(rng, 128, 8192), _log(rng, 1, 64)
        shape = rng.choice(["any", "any", "k64", "k128"])  # any size, or inputs of whole segments
        if kind == "int4" or shape == "k128":
            k = 128 * max(1, k // 128)
        elif shape == "k64":
            k = 64 * max(1, k // 64)
        return {"path": "linear", "kind": kind, "n": n, "k": k, "rows": rows, "bias": rng.random() < 0.3}
    if path == "linears":
        return {"path": "linears", "kind": kind, "hidden": 128 * rng.randint(4, 18), "ffn": 128 * rng.randint(12, 66),
                "layers": rng.randint(1, 4), "rows": _log(rng, 1, 64)}
    if path == "attention":
        head_dim = rng.choice([64, 128, 128])
        max_len = rng.choice([512, 1024, 2048, 4096])
        rows = rng.choice([1, 1, rng.randint(2, 16)])
        return {"path": "attention", "heads": rng.randint(4, 20), "head_dim": head_dim, "layers": rng.randint(2, 8),
                "rows": rows, "pos": _log(rng, 8, max_len - rows), "max_len": max_len}
    if path in ("round", "steps"):
        nh, dq, dv = rng.choice([(16, 64, 128), (4, 256, 256), (rng.randint(2, 16), rng.choice([64, 128, 192, 256]),
                                                                4 * rng.randint(8, 64))])
        t = _log(rng, 2, 40) if path == "round" else rng.randint(2, 20)
        case = {"path": path, "dtype": rng.choice(["bf16", "bf16", "fp32", "fp16"]), "nh": nh, "dq": dq, "dv": dv,
                "t": t, "accepted": rng.randint(0, t - 1)}
        if path == "round":
            case["layers"] = rng.randint(1, 6)
        return case
    heads = rng.choice([8, 16])
    case = {"path": rng.choice(["step", "verify", "prompt"]), "kind": kind, "hidden": 128 * heads,
            "ffn": 512 * rng.randint(4, 16), "heads": heads, "layers": rng.randint(2, 8),
            "vocab": rng.choice([8192, 32768, 100352])}
    if case["path"] == "prompt":
        case["tokens"] = _log(rng, 8, 320)
    else:
        case["pos"] = _log(rng, 4, 1000)
        if case["path"] == "verify":
            case["rows"] = rng.randint(2, 16)
    return case


# --- inputs ---------------------------------------------------------------------------------------------------------


def _gen(seed: int) -> torch.Generator:
    return torch.Generator(device=DEV).manual_seed(int(seed))


def _randn(g: torch.Generator, *shape: int, std: float = 1.0, dtype=BF) -> torch.Tensor:
    return (torch.randn(*shape, generator=g, device=DEV) * std).to(dtype)


def _dequantized(kind: str, w: torch.Tensor, scale_dtype=BF) -> torch.Tensor:
    """float64 weights that a stored format of w [N, K] stands for: bf16 as they are; int8 per row (scale = max|row| /
    127 in the scale dtype, codes rounded to nearest even); int4 per row and 128 inputs (scale = (max - min) / 15
    stored as bf16, zero = -min / scale stored as fp16, codes 0..15)."""
    if kind == "bf16":
        return w.double()
    wf = w.float()
    if kind == "int8":
        floor = 2.0 ** -24 if scale_dtype == torch.float16 else 1e-12
        s = (wf.abs().amax(dim=1) / 127.0).clamp_min(floor).to(scale_dtype).float()
        return torch.round(wf / s[:, None]).clamp_(-127, 127).double() * s.double()[:, None]
    g = wf.reshape(w.shape[0], -1, 128)
    lo, hi = g.amin(-1), g.amax(-1)
    s = ((hi - lo) / 15.0).clamp_min(1e-6).to(BF).float()
    z = (-lo / s).to(torch.float16).float()
    codes = torch.round(g / s[..., None] + z[..., None]).clamp_(0, 15)
    return ((codes.double() - z.double()[..., None]) * s.double()[..., None]).reshape(w.shape)


def _linear_inputs(case: dict, seed: int):
    g = _gen(seed)
    w = _randn(g, case["n"], case["k"], std=0.02)
    b = _randn(g, case["n"], std=0.02) if case["bias"] else None
    x = _randn(g, case["rows"], case["k"])
    return w, b, x


def _linears_inputs(case: dict, seed: int):
    g = _gen(seed)
    dim = {"h": case["hidden"], "f": case["ffn"]}
    ws = [[_randn(g, dim[n], dim[k], std=0.02) for _, n, k in ROLES] for _ in range(case["layers"])]
    xs = [_randn(g, case["rows"], dim[k]) for _, _, k in ROLES]
    xs[1] = xs[2] = xs[0]  # q, k, v share their input, gate and up theirs
    xs[5] = xs[4]
    return ws, xs


def _attention_inputs(case: dict, seed: int) -> list[dict]:
    g = _gen(seed)
    hd, d = case["heads"], case["head_dim"]
    return [{"qkv": _randn(g, case["rows"], 3 * hd * d),
             "qw": (1.0 + _randn(g, hd * d, std=0.1, dtype=torch.float32)).to(BF),
             "kw": (1.0 + _randn(g, hd * d, std=0.1, dtype=torch.float32)).to(BF),
             "kc": _randn(g, hd, case["max_len"], d), "vc": _randn(g, hd, case["max_len"], d)}
            for _ in range(case["layers"])]


def _inv_freq(d: int, theta: float = 500000.0) -> torch.Tensor:
    return (1.0 / (theta ** (torch.arange(0, d, 2, dtype=torch.float) / d))).to(DEV)


def _mlstm_inputs(case: dict, seed: int) -> list[dict]:
    """Per layer: q, k (scaled by 1 / sqrt(dq)), v, gate pre-activations i ~ N(0, 1) and f ~ N(3, 1), a start state."""
    g = _gen(seed)
    t, nh, dq, dv, dt = case["t"], case["nh"], case["dq"], case["dv"], DTYPES[case["dtype"]]
    f32 = torch.float32
    return [{"q": _randn(g, t, nh, dq, dtype=dt), "k": _randn(g, t, nh, dq, std=dq ** -0.5, dtype=dt),
             "v": _randn(g, t, nh, dv, dtype=dt), "i": _randn(g, t, nh, 1, dtype=f32),
             "f": 3.0 + _randn(g, t, nh, 1, dtype=f32), "c": _randn(g, 1, nh, dq, dv, std=0.1, dtype=f32),
             "n": _randn(g, 1, nh, dq, std=0.1, dtype=f32), "m": _randn(g, 1, nh, 1, dtype=f32)}
            for _ in range(case.get("layers", 1))]


def _config(case: dict) -> olmo.OlmoConfig:
    return olmo.OlmoConfig(hidden=case["hidden"], ffn=case["ffn"], layers=case["layers"], heads=case["heads"],
                           vocab=case["vocab"])


def _model_weights(case: dict, seed: int) -> dict[str, torch.Tensor]:
    """bf16 weights in the decoder's key layout: linears ~ N(0, 4 / hidden), norms ~ 1 + N(0, 0.1^2), embeddings
    ~ N(0, 1)."""
    g = _gen(seed)
    h, f, v = case["hidden"], case["ffn"], case["vocab"]
    std = 2.0 / h ** 0.5

    def norm() -> torch.Tensor:
        return (1.0 + _randn(g, h, std=0.1, dtype=torch.float32)).to(BF)

    w = {"embed": _randn(g, v, h)}
    for layer in range(case["layers"]):
        p = f"l{layer}."
        for name in ("q", "k", "v", "o"):
            w[p + name] = _randn(g, h, h, std=std)
        w[p + "gate"], w[p + "up"], w[p + "down"] = (_randn(g, f, h, std=std), _randn(g, f, h, std=std),
                                                     _randn(g, h, f, std=std))
        for name in ("q_norm", "k_norm", "post_attn", "post_ff"):
            w[p + name] = norm()
    w["norm"], w["lm_head"] = norm(), _randn(g, v, h, std=std)
    return w


def _model_tokens(case: dict, seed: int) -> torch.Tensor:
    count = case["tokens"] if case["path"] == "prompt" else case.get("rows", 1)
    return torch.randint(0, case["vocab"], (count,), generator=_gen(seed + 7919), device=DEV)


def _model_caches(case: dict, seed: int):
    """What earlier positions left in the caches: [layers, heads, pos, head_dim]."""
    g = _gen(seed + 104729)
    shape = (case["layers"], case["heads"], case["pos"], case["hidden"] // case["heads"])
    return _randn(g, *shape), _randn(g, *shape)


def _capture(fn) -> torch.cuda.CUDAGraph:
    """fn warmed up on a side stream and captured, as the decode loops capture their steps."""
    s = torch.cuda.Stream()
    s.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(s):
        for _ in range(2):
            fn()
    torch.cuda.current_stream().wait_stream(s)
    torch.cuda.synchronize()
    g = torch.cuda.CUDAGraph()
    with torch.cuda.graph(g):
        fn()
    return g


# --- prepare and run ------------------------------------------------------------------------------------------------


def _module(w: torch.Tensor, b: torch.Tensor | None, kind: str, rows: int) -> nn.Module:
    lin = nn.Linear(w.shape[1], w.shape[0], bias=b is not None, device="meta", dtype=BF)
    lin.weight = nn.Parameter(w, requires_grad=False)
    if b is not None:
        lin.bias = nn.Parameter(b, requires_grad=False)
    if kind == "int8" and rows == 1:  # the one-row layer; more rows go through the skinny one
        return Int8Linear(lin)
    return SkinnyLinear(lin, f"{kind}_wo")


def _prepare_linear(case, seed):
    w, b, x = _linear_inputs(case, seed)
    return {"layer": _module(w, b, case["kind"], case["rows"]), "x": x}


def _run_linear(s):
    return s["layer"](s["x"])


def _prepare_linears(case, seed):
    ws, xs = _linears_inputs(case, seed)
    layers = [[SkinnyLinear(_linear_of(w), f"{case['kind']}_wo") for w in ws.pop(0)] for _ in range(case["layers"])]
    s: dict = {"layers": layers, "xs": xs}

    def fn():
        s["out"] = [[lin(x) for lin, x in zip(layer, xs)] for layer in layers]

    s["graph"] = _capture(fn)
    return s


def _linear_of(w: torch.Tensor) -> nn.Linear:
    lin = nn.Linear(w.shape[1], w.shape[0], bias=False, device="meta", dtype=BF)
    lin.weight = nn.Parameter(w, requires_grad=False)
    return lin


def _run_graph(s):
    s["graph"].replay()
    return s["out"]


def _prepare_attention(case, seed):
    layers = _attention_inputs(case, seed)
    hd, d, rows, pos = case["heads"], case["head_dim"], case["rows"], case["pos"]
    inv = _inv_freq(d)
    pos_t = torch.tensor([pos], dtype=torch.int64, device=DEV)
    outs = [torch.empty(rows, hd * d, dtype=BF, device=DEV) for _ in layers]
    lib = _lib.lib()

    def fn():
        st = torch.cuda.current_stream().cuda_stream
        for w, out in zip(layers, outs):
            rc = lib.bp_decode_rope_attention_rows(w["qkv"].data_ptr(), w["qw"].data_ptr(), w["kw"].data_ptr(),
                                                   inv.data_ptr(), pos_t.data_ptr(), w["kc"].data_ptr(),
                                                   w["vc"].data_ptr(), out.data_ptr(), hd, d, rows, case["max_len"],
                                                   EPS, d ** -0.5, st)
            _lib.check(rc, "bp_decode_rope_attention_rows")

    written = [(w["kc"][:, pos:pos + rows], w["vc"][:, pos:pos + rows]) for w in layers]
    return {"inputs": (layers, inv, pos_t), "graph": _capture(fn), "out": {"attn": outs, "written": written}}


def _prepare_round(case, seed):
    t, nh, dq, dv, acc = case["t"], case["nh"], case["dq"], case["dv"], case["accepted"]
    inputs = _mlstm_inputs(case, seed)
    # the layers' states as views of one buffer, so that one copy puts the start states back before a pass
    sizes = [nh * dq * dv, nh * dq, nh]
    start = torch.cat([p[k].reshape(-1) for p in inputs for k in ("c", "n", "m")])
    live = start.clone()
    states, at = [], 0
    for _ in inputs:
        views = []
        for size, shape in zip(sizes, ((1, nh, dq, dv), (1, nh, dq), (1, nh, 1))):
            views.append(live[at:at + size].view(shape))
            at += size
        states.append(tuple(views))
    hs = [torch.zeros(t, nh, dv, dtype=p["q"].dtype, device=DEV) for p in inputs]
    saved = [(torch.zeros(nh, dq, device=DEV), torch.zeros(nh, device=DEV)) for _ in inputs]
    tok = torch.arange(100, 100 + t, dtype=torch.int64, device=DEV)
    ids = torch.cat([tok.new_zeros(1), tok])[:t].contiguous()
    if acc + 1 < t:
        ids[acc + 1] = 1  # the first rejected draft
    verdict = torch.zeros(t + 1, dtype=torch.int64, device=DEV)
    length = verdict[t]

    def fn():
        live.copy_(start)
        for p, cur, h, (ns, ms) in zip(inputs, states, hs, saved):
            draft_fused.multistep_fw(cur, p["q"], p["k"], p["v"], p["i"], p["f"], h, ns, ms, EPS)
        draft_fused.accept(ids, tok, verdict, t, t)
        for p, cur, (ns, ms) in zip(inputs, states, saved):
            draft_fused.lazy_commit(cur, p["k"], p["v"], p["i"], p["f"], length, ns, ms)

    return {"inputs": (inputs, start, tok, ids, saved), "graph": _capture(fn),
            "out": {"h": hs, "state": states, "verdict": verdict}}


def _prepare_steps(case, seed):
    t, nh, dq, dv, acc = case["t"], case["nh"], case["dq"], case["dv"], case["accepted"]
    p = _mlstm_inputs(case, seed)[0]
    hist = tuple(x.expand(t + 1, *x.shape).contiguous() for x in (p["c"], p["n"], p["m"]))  # slot 0: the start
    cur = tuple(torch.zeros_like(x) for x in (p["c"], p["n"], p["m"]))
    h = torch.zeros(t, nh, dv, dtype=p["q"].dtype, device=DEV)
    length = torch.tensor(acc + 1, dtype=torch.int64, device=DEV)  # the slot after position `accepted`

    def fn():
        for j in range(t):
            draft_core.mlstm_step_into(tuple(x[j] for x in hist), tuple(x[j + 1] for x in hist), p["q"][j:j + 1],
                                       p["k"][j:j + 1], p["v"][j:j + 1], p["i"][j:j + 1], p["f"][j:j + 1],
                                       h[j:j + 1], EPS)
        draft_core.commit_state(hist, cur, length)

    return {"inputs": (p, length), "graph": _capture(fn), "out": {"h": h, "state": cur, "history": hist}}


def _prepare_model(case, seed):
    dec = olmo.OlmoDecoder(_config(case), _model_weights(case, seed), case["kind"])
    ids = _model_tokens(case, seed)
    if case["path"] == "prompt":
        return {"dec": dec, "ids": ids.cpu()[None], "generate": olmo.make_generate_graph(dec)}
    pos, rows = case["pos"], case.get("rows", 1)
    kc, vc = _model_caches(case, seed)
    dec.k_cache[:, :, :pos], dec.v_cache[:, :, :pos] = kc, vc
    s: dict = {"dec": dec, "ids": ids, "pos": pos}
    if case["path"] == "step":
        s["graph"] = _capture(lambda: (dec.tok.copy_(ids), dec.pos.fill_(pos), dec.step()))
        s["out"] = {"logits": dec.logits, "pos": dec.pos, "k": dec.k_cache[:, :, pos:pos + 1],
                    "v": dec.v_cache[:, :, pos:pos + 1]}
        return s
    dec.verify_buffers(rows)
    s["graph"] = _capture(lambda: (dec.v_ids[:rows].copy_(ids), dec.v_pos.fill_(pos), dec.verify(rows)))
    s["out"] = {"logits": dec.vlogits[:rows], "pos": dec.v_pos, "k": dec.k_cache[:, :, pos:pos + rows],
                "v": dec.v_cache[:, :, pos:pos + rows]}
    return s


def _run_prompt(s):
    tokens = s["generate"](s["ids"], max_new_tokens=1)
    dec, n = s["dec"], s["ids"].shape[1]
    return {"logits": dec.logits, "tokens": tokens, "k": dec.k_cache[:, :, :n], "v": dec.v_cache[:, :, :n]}


_PREPARE = {"linear": _prepare_linear, "linears": _prepare_linears, "attention": _prepare_attention,
            "round": _prepare_round, "steps": _prepare_steps, "step": _prepare_model, "verify": _prepare_model,
            "prompt": _prepare_model}


def prepare(case: dict, seed: int) -> dict:
    s = _PREPARE[case["path"]](case, seed)
    s["run"] = {"linear": _run_linear, "prompt": _run_prompt}.get(case["path"], _run_graph)
    return s


@torch.no_grad()
def run(state: dict):
    return state["run"](state)


# --- work and tolerance ---------------------------------------------------------------------------------------------


def _weight_bytes(kind: str, n: int, k: int) -> float:
    return {"bf16": 2.0 * n * k, "int8": n * k + 2.0 * n, "int4": 0.5 * n * k + 4.0 * n * k / 128}[kind]


def work(case: dict) -> dict:
    path = case["path"]
    if path == "linear":
        n, k, m = case["n"], case["k"], case["rows"]
        return {"bytes": _weight_bytes(case["kind"], n, k) + 2.0 * m * (n + k) + 2.0 * n * case["bias"],
                "flops": 2.0 * m * n * k}
    if path == "linears":
        h, f, m, count = case["hidden"], case["ffn"], case["rows"], case["layers"]
        w = 4 * _weight_bytes(case["kind"], h, h) + 2 * _weight_bytes(case["kind"], f, h) \
            + _weight_bytes(case["kind"], h, f)
        return {"bytes": count * (w + 2.0 * m * (5 * h + 2 * f)) + 2.0 * m * (3 * h + f),
                "flops": count * 2.0 * m * (4 * h * h + 3 * h * f)}
    if path == "attention":
        h, m, t = case["heads"] * case["head_dim"], case["rows"], case["pos"] + case["rows"]
        return {"bytes": case["layers"] * 2.0 * (2 * t * h + 4 * m * h + 2 * m * h + 2 * h),
                "flops": case["layers"] * 4.0 * m * t * h}
    if path in ("round", "steps"):
        nh, dq, dv, t, io = case["nh"], case["dq"], case["dv"], case["t"], 4 if case["dtype"] == "fp32" else 2
        state = 4.0 * nh * (dq * dv + dq + 1)
        rows = float(t * nh) * (io * (2 * dq + 2 * dv) + 8)
        flops = 8.0 * t * nh * dq * dv
        if path == "steps":  # the history is part of the result: a state per position, and the committed one
            return {"bytes": rows + (t + 2) * state, "flops": flops}
        return {"bytes": case["layers"] * (rows + 2 * state), "flops": case["layers"] * 2.0 * flops}
    h, f, v, nl = case["hidden"], case["ffn"], case["vocab"], case["layers"]
    m = case["tokens"] if path == "prompt" else case.get("rows", 1)
    ctx = m if path == "prompt" else case["pos"] + m  # cache positions read or written
    heads_rows = 1 if path == "prompt" else m  # a prompt needs its last position's logits only
    w = nl * (4 * _weight_bytes(case["kind"], h, h) + 3 * _weight_bytes(case["kind"], f, h)) \
        + _weight_bytes(case["kind"], v, h)
    seen = m * (m + 1) / 2 if path == "prompt" else m * ctx
    return {"bytes": w + nl * 4.0 * ctx * h + 2.0 * m * h + 2.0 * heads_rows * v,
            "flops": 2.0 * m * nl * (4 * h * h + 3 * f * h) + 2.0 * heads_rows * v * h + 4.0 * nl * seen * h}


def tolerance(case: dict) -> dict:
    """About four times the error of the path against float64, measured once."""
    path = case["path"]
    if path in ("linear", "linears"):  # 1.7e-3: one bf16 rounding of a 32-bit sum; 2.4e-3 with the bias added after it
        return {"rel": 8e-3, "max": 2e-2}
    if path == "attention":  # 6e-3: q, k and the probabilities rounded to bf16, one rounding of the result
        return {"rel": 2.5e-2, "max": 1.5e-1}
    if path in ("round", "steps"):
        # 32-bit recurrences 1e-7 (a normaliser near its bound magnifies their rounding in an output); 16 bits: the
        # rounded gates, state operands and outputs, 3.5e-3 in bf16 and 4.3e-4 in fp16
        return {"fp32": {"rel": 1e-5, "max": 1e-3}, "bf16": {"rel": 1.4e-2, "max": 3e-1},
                "fp16": {"rel": 2e-3, "max": 5e-2}}[case["dtype"]]
    # whole models, 1.1e-2 to 2.4e-2: a different rounding anywhere travels through every later layer in bf16
    return {"rel": 3e-2, "max": 3e-1, "differ": 1e-2}


# --- the same in float64 --------------------------------------------------------------------------------------------


def _exact_linears(case, seed):
    ws, xs = _linears_inputs(case, seed)
    return [[x.double() @ _dequantized(case["kind"], w).T for w, x in zip(layer, xs)] for layer in ws]


def _rms(x: torch.Tensor, w: torch.Tensor) -> torch.Tensor:
    return x * torch.rsqrt(x.square().mean(-1, keepdim=True) + EPS) * w.double()


def _rope(x: torch.Tensor, pos0: int, inv: torch.Tensor) -> torch.Tensor:
    """x [rows, heads, d] rotated at positions pos0, pos0 + 1, ..."""
    a = (torch.arange(pos0, pos0 + x.shape[0], device=DEV, dtype=torch.float64)[:, None] * inv.double())[:, None]
    lo, hi = x.chunk(2, -1)
    return torch.cat([lo * a.cos() - hi * a.sin(), hi * a.cos() + lo * a.sin()], -1)


def _exact_attention_layer(qkv, qw, kw, kc, vc, pos, heads, inv):
    """Rows at pos .. over cached k, v [heads, pos, d] and themselves: (out [rows, h], k, v [heads, rows, d])."""
    rows, d = qkv.shape[0], qkv.shape[1] // 3 // heads
    q, k, v = qkv.chunk(3, -1)
    q = _rope(_rms(q, qw).view(rows, heads, d), pos, inv).transpose(0, 1)
    k = _rope(_rms(k, kw).view(rows, heads, d), pos, inv).transpose(0, 1)
    v = v.view(rows, heads, d).transpose(0, 1)
    keys, vals = torch.cat([kc, k], 1), torch.cat([vc, v], 1)
    s = torch.matmul(q, keys.transpose(1, 2).contiguous()) * d ** -0.5
    late = torch.arange(keys.shape[1], device=DEV)[None] > pos + torch.arange(rows, device=DEV)[:, None]
    p = s.masked_fill(late, -math.inf).softmax(-1)
    return torch.matmul(p, vals).transpose(0, 1).reshape(rows, heads * d), k, v


def _exact_attention(case, seed):
    inv, pos = _inv_freq(case["head_dim"]), case["pos"]
    outs, written = [], []
    for w in _attention_inputs(case, seed):
        out, k, v = _exact_attention_layer(w["qkv"].double(), w["qw"], w["kw"], w["kc"][:, :pos].double(),
                                           w["vc"][:, :pos].double(), pos, case["heads"], inv)
        outs.append(out)
        written.append((k, v))
    return {"attn": outs, "written": written}


def _exact_recurrence(p: dict):
    """h of every position and the state after each."""
    q, k, v, i, f = (p[n].double() for n in "qkvif")
    c, n, m = p["c"][0].double(), p["n"][0].double(), p["m"][0, :, 0].double()
    hs, states = [], [(c, n, m)]
    for t in range(q.shape[0]):
        fl, it = torch.nn.functional.logsigmoid(f[t, :, 0]), i[t, :, 0]
        mn = torch.maximum(fl + m, it)
        fa, ia, m = torch.exp(fl + m - mn), torch.exp(it - mn), mn
        c = fa[:, None, None] * c + ia[:, None, None] * k[t][:, :, None] * v[t][:, None]
        n = fa[:, None] * n + ia[:, None] * k[t]
        qs = q[t] * q.shape[-1] ** -0.5
        num = (qs[:, :, None] * c).sum(1)
        den = torch.maximum((qs * n).sum(-1).abs(), torch.exp(-m)) + EPS
        hs.append(num / den[:, None])
        states.append((c, n, m))
    return torch.stack(hs), states


def _exact_mlstm(case, seed):
    hs, cur, hist = [], [], None
    for p in _mlstm_inputs(case, seed):
        h, states = _exact_recurrence(p)
        hs.append(h)
        c, n, m = states[case["accepted"] + 1]
        cur.append((c[None], n[None], m[None, :, None]))
        hist = tuple(torch.stack([s[j] for s in states])[:, None] for j in range(3))
    if case["path"] == "steps":
        return {"h": hs[0], "state": cur[0], "history": (hist[0], hist[1], hist[2][..., None])}
    return {"h": hs, "state": cur, "verdict": None}


def _exact_model(case, seed):
    w, ids = _model_weights(case, seed), _model_tokens(case, seed)
    heads, nl = case["heads"], case["layers"]
    d = case["hidden"] // heads
    inv = _inv_freq(d)
    if case["path"] == "prompt":
        pos = 0
        kc = vc = torch.zeros(nl, heads, 0, d, device=DEV)
    else:
        pos = case["pos"]
        kc, vc = _model_caches(case, seed)
    scale_dtype = torch.float16  # the decoder's int8 scales

    def lin(x, name):
        return x @ _dequantized(case["kind"], w[name], scale_dtype).T

    x = w["embed"][ids].double()
    ks, vs = [], []
    for layer in range(nl):
        p = f"l{layer}."
        qkv = torch.cat([lin(x, p + n) for n in ("q", "k", "v")], -1)
        a, k, v = _exact_attention_layer(qkv, w[p + "q_norm"], w[p + "k_norm"], kc[layer].double(),
                                         vc[layer].double(), pos, heads, inv)
        ks.append(k)
        vs.append(v)
        x = x + _rms(lin(a, p + "o"), w[p + "post_attn"])
        x = x + _rms(lin(torch.nn.functional.silu(lin(x, p + "gate")) * lin(x, p + "up"), p + "down"),
                     w[p + "post_ff"])
    if case["path"] == "prompt":
        x = x[-1:]
    logits = lin(_rms(x, w["norm"]), "lm_head")
    whole = "tokens" if case["path"] == "prompt" else "pos"
    return {"logits": logits, whole: None, "k": torch.stack(ks), "v": torch.stack(vs)}


def _exact_linear(case, seed):
    w, b, x = _linear_inputs(case, seed)
    y = x.double() @ _dequantized(case["kind"], w).T
    return y if b is None else y + b.double()


@torch.no_grad()
def exact(case: dict, seed: int):
    path = case["path"]
    if path == "linear":
        return _exact_linear(case, seed)
    if path == "linears":
        return _exact_linears(case, seed)
    if path == "attention":
        return _exact_attention(case, seed)
    if path in ("round", "steps"):
        return _exact_mlstm(case, seed)
    return _exact_model(case, seed)
