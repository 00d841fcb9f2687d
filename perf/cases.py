"""The calls a program that serves tokens makes of this library, as timed cases.

Every case goes through the C ABI of include/ultima_hsamp.h as a serving loop
binds it: one sampler handle for the whole program, the batch descriptors
filled once, one call per step on the current stream. Five kinds:

  sample  ultima_hsamp_run over [rows, vocab] logits on the device
  decode  ultima_hsamp_run_commit: the server's step over many slots, their
          histories kept and appended on the device
  verify  ultima_hsamp_verify_block: a drafted block against the target's logits
  host    ultima_hsamp_sample_host: sample() on one row in host memory, the
          logits left as sample() leaves them
  head    ultima_hsamp_lm_head: final norm, optional fold, lm-head product

`knobs` names the sampling parameters of a batch; KNOBS below.
"""
import ctypes
import importlib.util
import math
import sys
from pathlib import Path

import numpy as np
import torch

PKG_DIR = Path(__file__).resolve().parent.parent / "ultima.cpp_amd"
V_QWEN = 151936
DECODE_STEPS = 512   # steps of a decode loop before a slot meets the same logits again


def _package():
    """ultima.cpp_amd as `ultima_cpp_amd` (the folder's name is no identifier)."""
    if "ultima_cpp_amd" not in sys.modules:
        spec = importlib.util.spec_from_file_location(
            "ultima_cpp_amd", PKG_DIR / "__init__.py", submodule_search_locations=[str(PKG_DIR)])
        mod = importlib.util.module_from_spec(spec)
        sys.modules["ultima_cpp_amd"] = mod
        spec.loader.exec_module(mod)
    return sys.modules["ultima_cpp_amd"]


WEIGHTS = ("bf16", "f32", "q4_k", "q5_k", "q6_k", "q8_0", "q4_1", "q5_0", "pq2_0")

# cli          SamplerParams::identity() with a temperature: the whole vocabulary, nothing cut
# server       SamplerParams{}: repetition 64, DRY 512, T .2, top-k 40, top-p .95, min-p .05
# penalties    repetition, frequency and presence over the whole history, T .7, top-k 50
# nucleus      top-p .9 over the whole vocabulary, nothing else
# constrained  a grammar's allowed-token mask, top-k 20, top-p .8
# mixed        every row its own temperature, top-k up to 1000, top-p and repetition penalty
# open         what a chat client sends with top-k off: repetition 1.1, T .8, top-p .95, min-p .05
# greedy       temperature 0 after a repetition penalty
KNOBS = ("cli", "server", "penalties", "nucleus", "constrained", "mixed", "open", "greedy")


def listed():
    def sample(name, knobs, rows, dtype="f32", hist=0, sets=False):
        return dict(name=name, kind="sample", knobs=knobs, rows=rows, vocab=V_QWEN, dtype=dtype, hist=hist,
                    bias=0, aligned=True, sets=sets)

    def head(name, weight, rows, fold=0):
        return dict(name=name, kind="head", weight=weight, rows=rows, hidden=4096, vocab=V_QWEN, fold=fold, scale=1.0)

    return [
        # one token of an interactive session: latency of a single row
        sample("cli_token", "cli", 1),
        # the drop-in's sample(): a host row in, the logits left in place
        dict(name="host_token", kind="host", knobs="server", vocab=V_QWEN, hist=600),
        # one step of a 64-slot server with the default parameters
        dict(name="decode_slots", kind="decode", knobs="server", rows=64, vocab=V_QWEN),
        # 16 chat sessions with top-k off: penalties, top-p and min-p over the whole vocabulary
        sample("open_slots", "open", 16, hist=600),
        # a batch with every penalty over long histories
        sample("batch_penalties", "penalties", 64, hist=2048),
        # nucleus sampling with no top-k: half the rows peaked, half nearly flat
        sample("batch_nucleus", "nucleus", 256),
        # constrained decoding, the kept ids and probabilities asked for
        sample("batch_constrained", "constrained", 128, dtype="bf16", sets=True),
        # 32 sequences of 32 candidate positions, each row its own parameters
        sample("batch_mixed", "mixed", 1024, dtype="bf16", hist=512),
        # the logits of one token: a bf16 head, and the usual quantised one
        head("head_bf16_token", "bf16", 1),
        head("head_q6k_token", "q6_k", 1),
        # a drafted block's logits from a quantised, folded head
        head("head_q4k_block", "q4_k", 16, fold=128),
        # a 64-slot step's logits
        head("head_bf16_slots", "bf16", 64),
    ]


def _log_int(rng, lo, hi):
    return min(hi, max(lo, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def draw(rng):
    """One more case of the ranges above: any kind and option, sizes over their
    logarithm, odd ones as they come."""
    kind = rng.choice(("sample", "sample", "sample", "head", "head", "decode", "verify", "host"))
    vocab = _log_int(rng, 8000, 262144)
    if kind == "head":
        weight = rng.choice(WEIGHTS)
        hidden = _log_int(rng, 512, 8192)
        if weight in ("bf16", "f32"):
            hidden = max(8, hidden // 8 * 8) if rng.random() < 0.75 else hidden
        else:
            hidden = max(256, hidden // 256 * 256)
        rows = _log_int(rng, 1, 64)
        vocab = min(vocab, 32 * V_QWEN * 4096 // (rows * hidden))
        fold = rng.choice((0, 0, 128)) if hidden % 128 == 0 else 0
        return dict(kind="head", weight=weight, rows=rows, hidden=hidden, vocab=vocab, fold=fold,
                    scale=rng.choice((1.0, 8.0)))
    if kind == "host":
        return dict(kind="host", knobs=rng.choice(("server", "cli", "open", "greedy")), vocab=vocab,
                    hist=_log_int(rng, 8, 2048))
    if kind == "decode":
        return dict(kind="decode", knobs=rng.choice(("server", "penalties", "greedy")), rows=_log_int(rng, 1, 256),
                    vocab=vocab)
    if kind == "verify":
        return dict(kind="verify", knobs=rng.choice(("server", "penalties")), rows=_log_int(rng, 2, 64), vocab=vocab,
                    dtype=rng.choice(("f32", "bf16")), hist=_log_int(rng, 8, 2048))
    knobs = rng.choice(KNOBS)
    dtype = rng.choice(("f32", "bf16"))
    rows = _log_int(rng, 1, 1024)
    if knobs in ("cli", "nucleus", "open"):
        rows = min(rows, max(1, 160 * V_QWEN // vocab), 256)
    else:
        rows = min(rows, max(1, 1024 * V_QWEN // vocab // (2 if dtype == "f32" else 1)))
    return dict(kind="sample", knobs=knobs, rows=rows, vocab=vocab, dtype=dtype,
                hist=_log_int(rng, 8, 2048) if knobs in ("server", "penalties", "mixed", "open", "greedy") else 0,
                bias=rng.choice((0, 0, 8)) if knobs in ("server", "penalties", "mixed") else 0,
                aligned=rng.random() < 0.6, sets=knobs in ("server", "penalties", "constrained", "mixed") and rng.random() < 0.5)


# ---- inputs ------------------------------------------------------------------------

def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(int(seed) & (2**62 - 1))


def _params(case, rows, seed):
    """One knob dict per row."""
    wl = _package().workloads
    knobs, hist = case["knobs"], case.get("hist", 0)
    one = {
        "cli": lambda: wl.identity_params(temperature=0.8),
        "server": wl.default_params,
        "penalties": lambda: wl.identity_params(temperature=0.7, top_k=50, rep_penalty=1.1, frequency_penalty=0.5,
                                                presence_penalty=0.3, repeat_last_n=hist or 512),
        "nucleus": lambda: wl.identity_params(top_p=0.9),
        "constrained": lambda: wl.identity_params(top_k=20, top_p=0.8),
        "open": lambda: wl.identity_params(temperature=0.8, top_p=0.95, min_p=0.05, rep_penalty=1.1, repeat_last_n=hist),
        "greedy": lambda: wl.identity_params(temperature=0.0, rep_penalty=1.1, repeat_last_n=hist or 64),
    }
    if knobs != "mixed":
        return [one[knobs]() for _ in range(rows)]
    r = np.random.default_rng(seed)
    t, p, q = r.uniform(0.2, 1.5, rows), r.uniform(0.5, 1.0, rows), r.uniform(1.0, 1.3, rows)
    k = r.integers(1, 1001, rows)
    return [wl.identity_params(temperature=float(np.float32(t[i])), top_k=int(k[i]), top_p=float(np.float32(p[i])),
                               rep_penalty=float(np.float32(q[i])), repeat_last_n=hist) for i in range(rows)]


def _logits(case, rows, vocab, g):
    """[rows, vocab] logits; nucleus batches: the first half N(0, 1) with 16
    tokens at +15, the rest N(0, 0.1^2)."""
    sigma = {"cli": 3.0, "server": 2.0, "penalties": 2.0, "constrained": 2.0, "mixed": 2.5, "open": 3.0,
             "greedy": 2.0, "nucleus": 1.0}[case["knobs"]]
    es = 2 if case.get("dtype") == "bf16" else 4
    stride = vocab if not case.get("aligned", True) else -(-vocab * es // 128) * 128 // es
    buf = torch.empty((rows, stride), dtype=torch.float32, device="cuda").normal_(0.0, sigma, generator=g)
    if case["knobs"] == "nucleus":
        half = (rows + 1) // 2
        at = torch.randint(0, vocab, (half, 16), generator=g, device="cuda")
        buf[:half].scatter_(1, at, 15.0)
        buf[half:] *= 0.1
    if es == 2:
        buf = buf.to(torch.bfloat16)
    return buf[:, :vocab]


def _mask(rows, vocab, g):
    """Allowed-token words (about 1% of the ids, at least one) and the same as booleans."""
    words = -(-vocab // 32)
    ok = torch.rand((rows, words * 32), generator=g, device="cuda") < 0.01
    ok[:, vocab:] = False
    ok.scatter_(1, torch.randint(0, vocab, (rows, 1), generator=g, device="cuda"), True)
    bit = torch.ones((), dtype=torch.int64, device="cuda") << torch.arange(32, device="cuda")
    w = (ok.view(rows, words, 32) * bit).sum(-1)
    return torch.where(w >= 2**31, w - 2**32, w).to(torch.int32), ok[:, :vocab]


def _inputs(case, seed):
    """What the call reads, made from the seed alone."""
    g = _generator(seed)
    i = {"kind": case["kind"]}
    if case["kind"] == "head":
        rows, H, V, t = case["rows"], case["hidden"], case["vocab"], case["weight"]
        i["hidden"] = torch.empty((rows, H), device="cuda").normal_(0.0, 2.0, generator=g)
        i["norm"] = torch.empty(H, device="cuda").normal_(1.0, 0.2, generator=g)
        i["signs"] = (torch.randint(0, 2, (H,), generator=g, device="cuda") * 2 - 1).float() if case["fold"] else None
        if t in ("bf16", "f32"):
            w = torch.empty((V, H), dtype=torch.bfloat16 if t == "bf16" else torch.float32, device="cuda")
            for a in range(0, V, 16384):
                n = min(16384, V - a)
                w[a:a + n] = torch.empty((n, H), device="cuda").normal_(0.0, 0.03, generator=g)
        else:
            be, bb, fields = _package().workloads.QUANT_BLOCKS[_weight_type(t)]
            nb = V * (H // be)
            w = torch.randint(0, 256, (nb, bb), generator=g, device="cuda", dtype=torch.uint8)
            for j, off in enumerate(fields):   # fp16 scales, and the smaller fp16 mins
                d = torch.rand(nb, generator=g, device="cuda") * (0.02 if j == 0 else 0.005)
                w[:, off:off + 2] = d.to(torch.float16).view(torch.uint8).view(nb, 2)
            w = w.view(V, H // be * bb)
        i["weight"] = w
        return i
    rows, V = (1 if case["kind"] == "host" else case["rows"]), case["vocab"]
    i["params"] = _params(case, rows, seed)
    # a decode loop's logits are new at every step: a window of `rows` rows that
    # moves down one row a step, so that a slot meets a row again only after as
    # many steps as its penalties look back
    i["logits"] = _logits(case, rows + (DECODE_STEPS if case["kind"] == "decode" else 0), V, g)
    i["u"] = torch.rand(rows, generator=g, device="cuda", dtype=torch.float64)
    i["mask"], i["allowed"] = _mask(rows, V, g) if case["knobs"] == "constrained" else (None, None)
    r = np.random.default_rng(seed + 1)
    i["bias"] = None
    if case.get("bias"):
        i["bias"] = [dict(zip(r.choice(V, case["bias"], replace=False).tolist(),
                              r.normal(0.0, 2.0, case["bias"]).astype(np.float32).tolist())) for _ in range(rows)]
    if case["kind"] == "decode":
        i["hist"] = torch.randint(0, V, (rows, 1024), generator=g, device="cuda", dtype=torch.int32)
        i["lens"] = torch.randint(1, 1024, (rows,), generator=g, device="cuda", dtype=torch.int32)
    elif case["kind"] == "verify":
        # the drafted ids (the target's most likely ones) follow the sequence's in memory
        h = torch.randint(0, V, (case["hist"],), generator=g, device="cuda", dtype=torch.int32)
        i["seq"] = torch.cat([h, i["logits"].float().argmax(1).to(torch.int32)])
    elif case.get("hist"):
        i["hist"] = torch.randint(0, V, (rows, case["hist"]), generator=g, device="cuda", dtype=torch.int32)
    return i


def _weight_type(t):
    hs = _package().hsamp
    return {"bf16": hs.BF16, "f32": hs.F32, "q4_k": hs.HEAD_Q4_K, "q5_k": hs.HEAD_Q5_K, "q6_k": hs.HEAD_Q6_K,
            "q8_0": hs.HEAD_Q8_0, "q4_1": hs.HEAD_Q4_1, "q5_0": hs.HEAD_Q5_0, "pq2_0": hs.HEAD_PQ2_0}[t]


# ---- the calls ---------------------------------------------------------------------

_handle = None


def _sampler():
    """The program's one sampler handle."""
    global _handle
    if _handle is None:
        _handle = _package().hsamp.Sampler(0, max_rows=1024, max_vocab=262144)
    return _handle


def _ptr(t):
    return None if t is None else t.data_ptr()


def prepare(case, seed):
    hs = _package().hsamp
    i = _inputs(case, seed)
    s = dict(i, lib=hs.lib())
    if case["kind"] == "head":
        rows, V = case["rows"], case["vocab"]
        s["logits"] = torch.empty((rows, V), device="cuda")
        s["normed"] = torch.empty((rows, case["hidden"]), device="cuda")
        h = hs.Head()
        h.hidden, h.hidden_stride, h.rows, h.hidden_dim, h.vocab = _ptr(i["hidden"]), case["hidden"], rows, case["hidden"], V
        h.weight_dtype, h.norm_scale, h.eps, h.logit_scale = _weight_type(case["weight"]), _ptr(i["norm"]), 1e-6, case["scale"]
        h.weight, h.normed, h.logits, h.logits_stride = _ptr(i["weight"]), _ptr(s["normed"]), _ptr(s["logits"]), V
        h.fold_block, h.fold_signs = case["fold"], _ptr(i["signs"])
        s["call"] = h
        return s
    s["handle"] = _sampler()
    rows, V = len(i["params"]), case["vocab"]
    if case["kind"] == "host":
        s["row"] = i["logits"][0].cpu().numpy()
        s["ids"] = i["hist"][0].cpu().numpy() if "hist" in i else None
        s["uniform"] = float(i["u"].cpu()[0])
        return s
    if case["kind"] == "verify":
        n = case["hist"]
        parr, _, _ = hs.make_params(i["params"][:1])
        s["work"] = torch.empty(int(s["lib"].ultima_hsamp_verify_work_ints(rows, n)), dtype=torch.int32, device="cuda")
        s["out"] = {k: torch.zeros(m, dtype=torch.int32, device="cuda")
                    for k, m in (("tokens", rows), ("count", 1), ("row_flags", rows))}
        v = hs.Verify()
        v.n_pos, v.vocab, v.dtype = rows, V, hs.F32 if case["dtype"] == "f32" else hs.BF16
        v.logits, v.logits_stride = _ptr(i["logits"]), i["logits"].stride(0)
        v.hist, v.hist_len, v.draft = _ptr(i["seq"]), n, i["seq"].data_ptr() + 4 * n
        v.u, v.params, v.work = _ptr(i["u"]), parr, _ptr(s["work"])
        v.out_tokens, v.out_count, v.row_flags = (_ptr(s["out"][k]) for k in ("tokens", "count", "row_flags"))
        s["call"], s["keep"] = v, parr
        return s
    out = {k: torch.zeros(rows, dtype=torch.int32, device="cuda") for k in ("token", "row_flags")}
    hist_len = [i["hist"].shape[1]] * rows if "hist" in i else [0] * rows
    if case["kind"] == "decode":
        hist_len = [0] * rows   # read on the device
        s["active"] = torch.ones(rows, dtype=torch.int32, device="cuda")
        s["budget"] = torch.full((rows,), 1 << 30, dtype=torch.int32, device="cuda")
        s["stop"] = np.array([151643, 151645], np.int32)
        c = hs.Commit()
        c.hist, c.hist_stride, c.hist_len_dev = _ptr(i["hist"]), i["hist"].stride(0), _ptr(i["lens"])
        c.active, c.budget, c.keep = _ptr(s["active"]), _ptr(s["budget"]), 512
        c.n_stop, c.stop_ids = 2, s["stop"].ctypes.data
        s["commit"] = c
    b, keep = s["handle"].batch(i["logits"][:rows], i["params"], i["u"], hist=i.get("hist"), hist_len=hist_len,
                                mask=i["mask"], bias=i["bias"], outputs=out)
    if case["kind"] == "decode":
        b.hist_len_dev = _ptr(i["lens"])
        s["at"] = 0
    if case["knobs"] == "nucleus" or case.get("sets"):
        out["kept_count"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        b.kept_count = _ptr(out["kept_count"])
    if case.get("sets"):
        b.set_cap = _cap(case)
        for k, dt in (("topk_idx", torch.int32), ("kept_idx", torch.int32), ("kept_prob", torch.float32)):
            out[k] = torch.zeros((rows, b.set_cap), dtype=dt, device="cuda")
            setattr(b, k, _ptr(out[k]))
        out["topk_count"] = torch.zeros(rows, dtype=torch.int32, device="cuda")
        b.topk_count = _ptr(out["topk_count"])
    s["call"], s["keep"], s["out"] = b, keep, out
    return s


def _cap(case):
    return 1024 if case["knobs"] == "mixed" else 64


def _stream():
    return ctypes.c_void_p(torch.cuda.current_stream().cuda_stream)


def run(state):
    hs, lib, kind = _package().hsamp, state["lib"], state["kind"]
    if kind == "head":
        hs.check(lib.ultima_hsamp_lm_head(ctypes.byref(state["call"]), _stream()), "lm_head")
        return {"logits": state["logits"], "normed": state["normed"]}
    if kind == "host":
        token, left = state["handle"].sample_host(state["row"], state["params"][0], hist=state["ids"],
                                                  u=state["uniform"], writeback=True)
        return {"token": token, "logits": left}
    h = state["handle"].h
    if kind == "verify":
        hs.check(lib.ultima_hsamp_verify_block(h, ctypes.byref(state["call"]), _stream()), "verify_block")
        return state["out"]
    if kind == "decode":
        state["at"] = (state["at"] + 1) % DECODE_STEPS
        state["call"].logits = state["logits"][state["at"]].data_ptr()
        hs.check(lib.ultima_hsamp_run_commit(h, ctypes.byref(state["call"]), ctypes.byref(state["commit"]), _stream()),
                 "run_commit")
        return dict(state["out"], hist=state["hist"], lens=state["lens"], active=state["active"], budget=state["budget"])
    hs.check(lib.ultima_hsamp_run(h, ctypes.byref(state["call"]), _stream()), "run")
    return state["out"]


# ---- what a pass cannot do without ---------------------------------------------------

def work(case):
    V = case["vocab"]
    if case["kind"] == "head":
        rows, H = case["rows"], case["hidden"]
        if case["weight"] in ("bf16", "f32"):
            row = H * (2 if case["weight"] == "bf16" else 4)
        else:
            row = _package().workloads.quant_row_bytes(_weight_type(case["weight"]), H)
        return {"bytes": V * row + rows * (2 * H + V) * 4 + H * (8 if case["fold"] else 4), "flops": 2.0 * rows * V * H}
    rows = 1 if case["kind"] == "host" else case["rows"]
    n = rows * V * (2 if case.get("dtype") == "bf16" else 4) + rows * (8 + 4 + 4)
    if case["kind"] == "host":
        n += V * 4 + case["hist"] * 4           # the logits come back
    elif case["kind"] == "decode":
        n += rows * (512 + 8) * 4
    else:
        n += rows * case["hist"] * 4
    if case["knobs"] == "constrained":
        n += rows * (-(-V // 32)) * 4
    return {"bytes": n, "flops": 0}


def tolerance(case):
    """Tokens, sets and counts are whole numbers and the same. Kept
    probabilities agree to 1e-6 (one float rounding per stage of a softmax over
    the same float logits); a head's logits are 32-bit sums of up to 8192
    products, whose order moves them by a few 1e-7 of their norm."""
    if case["kind"] == "head":
        return {"rel": 2e-6, "max": 2e-5}
    if case["kind"] == "host" or case.get("sets"):
        return {"rel": 1e-6, "max": 1e-6}
    return "exact"


# ---- the same in 64 bits -------------------------------------------------------------

def _final_logits(i, r, params, ids, V):
    """Row r's logits after mask, bias, penalties and temperature, in float64."""
    x = i["logits"][r].double().clone()
    if i["allowed"] is not None:
        x[~i["allowed"][r]] = -math.inf
    if i["bias"] is not None:
        for t, v in i["bias"][r].items():
            x[t] += v

    def counts(n):
        w = ids[-n:] if n and ids is not None else torch.zeros(0, dtype=torch.int64, device="cuda")
        return torch.bincount(w.long(), minlength=V).double()

    f = lambda k: float(np.float32(params[k]))  # noqa: E731
    if f("rep_penalty") != 1.0:
        seen = counts(params["repeat_last_n"]) > 0
        x = torch.where(seen, torch.where(x > 0, x / f("rep_penalty"), x * f("rep_penalty")), x)
    if f("dry_multiplier") > 0:
        c = counts(params["dry_last_n"])
        over = c - params["dry_allowed_len"]
        x = torch.where(over > 0, x - f("dry_multiplier") * f("dry_base") ** over.clamp(min=0), x)
    if f("frequency_penalty") or f("presence_penalty"):
        c = counts(max(params["repeat_last_n"], params["dry_last_n"]))
        x = torch.where(c > 0, x - c * f("frequency_penalty") - f("presence_penalty"), x)
    return x / f("temperature") if f("temperature") > 0 else x


def _kept(x, params):
    """(ids in index order, their probabilities, the logits left) after top-k, top-p and min-p."""
    order = torch.sort(x, descending=True, stable=True).indices
    k = params["top_k"]
    order = order[:k] if 0 < k < x.numel() else order
    order = order[x[order] > -math.inf]
    p = torch.softmax(x[order], 0)
    top_p, min_p = float(np.float32(params["top_p"])), float(np.float32(params["min_p"]))
    if 0 < top_p < 1:
        n = min(p.numel(), int((torch.cumsum(p, 0) < top_p).sum()) + 1)
        order, p = order[:n], torch.softmax(x[order[:n]], 0)
    if min_p > 0:
        order = order[p >= min_p * p.max()]
    ids = torch.sort(order).values
    left = torch.full_like(x, -math.inf)
    left[ids] = x[ids]
    return ids, torch.softmax(x[ids], 0), left


def _dequant(w, t, H):
    """float64 weights [M, H] of GGUF blocks."""
    be, bb, fields = _package().workloads.QUANT_BLOCKS[_weight_type(t)]
    b = w.view(-1, H // be, bb)
    f16 = lambda o: b[..., o:o + 2].contiguous().view(torch.float16).double()  # noqa: E731  ([..., 1])
    q = b.to(torch.int32)
    i8 = lambda v: torch.where(v > 127, v - 256, v)  # noqa: E731
    if t == "q8_0":
        out = i8(q[..., 2:34]) * f16(0)
    elif t == "q4_1":
        out = torch.cat([q[..., 4:20] & 15, q[..., 4:20] >> 4], -1) * f16(0) + f16(2)
    elif t == "q5_0":
        bit = (q[..., 2:6, None] >> torch.arange(8, device="cuda", dtype=torch.int32) & 1).flatten(-2)
        out = ((torch.cat([q[..., 6:22] & 15, q[..., 6:22] >> 4], -1) | bit << 4) - 16) * f16(0)
    elif t == "pq2_0":
        out = (torch.stack([q[..., 2:34] >> 2 * j & 3 for j in range(4)], -1).flatten(-2) - 1) * f16(0)
    elif t in ("q4_k", "q5_k"):
        s, parts = q[..., 4:16], []
        for j in range(8):
            sc = s[..., j] & 63 if j < 4 else s[..., j + 4] & 15 | s[..., j - 4] >> 6 << 4
            mn = s[..., j + 4] & 63 if j < 4 else s[..., j + 4] >> 4 | s[..., j] >> 6 << 4
            o = (16 if t == "q4_k" else 48) + 32 * (j // 2)
            v = q[..., o:o + 32] >> 4 * (j % 2) & 15
            if t == "q5_k":
                v = v | (q[..., 16:48] >> j & 1) << 4
            parts.append(v * (f16(0) * sc[..., None]) - f16(2) * mn[..., None])
        out = torch.cat(parts, -1)
    else:
        parts = []
        for j in range(8):
            half, run_ = j // 4, j % 4
            lo = q[..., 64 * half + 32 * (run_ % 2):64 * half + 32 * (run_ % 2) + 32] >> 4 * (run_ // 2) & 15
            v = lo | (q[..., 128 + 32 * half:160 + 32 * half] >> 2 * run_ & 3) << 4
            sc = i8(q[..., 192 + 8 * half + 2 * run_:194 + 8 * half + 2 * run_]).repeat_interleave(16, -1)
            parts.append((v - 32) * (f16(208) * sc))
        out = torch.cat(parts, -1)
    return out.reshape(-1, H)


def exact(case, seed):
    if case["kind"] != "head" and case["kind"] != "host" and not case.get("sets"):
        return None
    i = _inputs(case, seed)
    if case["kind"] == "head":
        H, V, t = case["hidden"], case["vocab"], case["weight"]
        x = i["hidden"].double()
        x = x * i["norm"].double() / torch.sqrt((x * x).mean(1, keepdim=True) + float(np.float32(1e-6)))
        if case["fold"]:
            x = (x * i["signs"].double()).view(-1, case["fold"])
            n = 1
            while n < case["fold"]:
                y = x.view(x.shape[0], -1, 2, n)
                x = torch.stack([y[:, :, 0] + y[:, :, 1], y[:, :, 0] - y[:, :, 1]], 2).view(x.shape[0], -1)
                n *= 2
            x = (x / math.sqrt(case["fold"])).view(-1, H)
        out = torch.empty((case["rows"], V), dtype=torch.float64, device="cuda")
        step = max(1, (1 << 26) // H)
        for a in range(0, V, step):
            w = i["weight"][a:a + step]
            w = w.double() if t in ("bf16", "f32") else _dequant(w, t, H)
            out[:, a:a + step] = x @ w.t().contiguous()
        return {"logits": out / case["scale"], "normed": x}
    V = case["vocab"]
    hist = i.get("hist")
    if case["kind"] == "host":
        x = _final_logits(i, 0, i["params"][0], None if hist is None else hist[0], V)
        if i["params"][0]["temperature"] <= 0:
            return {"token": None, "logits": x.cpu().numpy()}
        return {"token": None, "logits": _kept(x, i["params"][0])[2].cpu().numpy()}
    prob = torch.zeros((case["rows"], _cap(case)), dtype=torch.float64, device="cuda")
    for r, p in enumerate(i["params"]):
        kept = _kept(_final_logits(i, r, p, None if hist is None else hist[r], V), p)[1]
        prob[r, :kept.numel()] = kept[:_cap(case)]
    return {"kept_prob": prob, **{k: None for k in ("token", "row_flags", "kept_count", "topk_idx", "kept_idx", "topk_count")}}
