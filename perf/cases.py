"""The workloads this framework is timed on: the INT4 LM head with its selection, selection over
caller-owned logits, speculative verify and the decode loop, through the public Python entry points.

listed() holds one case for each kind of call a serving program makes, from the smallest to the
largest; draw() gives more cases of the same ranges. The ranges: heads of 32,000 to 262,144
vocabulary rows (any number, odd ones included) by d_model 1,024 to 5,376 (multiples of 128); 1 to
64 rows per call; histories of up to 4,096 ids; shortlists of 1 to 4,096 entries (top_k, 0 = none);
1 to 8 drafts per verify; generations of 8 to 32 tokens.

Weights are normal rows quantised to 4 bits per group of 64 (scale and bias per group from the
group's range), hidden rows are normal, softcap 30: the softmax of a row then puts about a fifth of
its mass on the best token, as a trained model's does.
"""
import importlib
import math

import numpy as np
import torch

twd = importlib.import_module("turbo-winfare-dense_amd")

DEV = "cuda:0"
CAP = 30.0
GROUP = 64
SIGMA = 0.28  # weight spread x sqrt(d / 30): logits of about 3.6 before the softcap
EPS = 1e-6
FULL_V, FULL_D = 262144, 5376


def listed():
    return [
        # one user decoding greedily: the latency of every token of a chat (the headline workload)
        {"name": "greedy_1_row", "kind": "greedy", "vocab": FULL_V, "d": FULL_D, "rows": 1},
        # the same on a small model with an odd vocabulary: the smallest head call, where launches
        # and the filling of the chip count
        {"name": "greedy_small_head", "kind": "greedy", "vocab": 32003, "d": 2048, "rows": 1},
        # a middle-sized batch on a vocabulary that ends in the middle of a tile: logits for a
        # program that picks its tokens itself
        {"name": "logits_24_rows", "kind": "logits", "vocab": 262143, "d": FULL_D, "rows": 24},
        # one user decoding with sampling and the repetition penalty over a long history
        {"name": "sample_1_row", "kind": "sample", "vocab": FULL_V, "d": FULL_D, "rows": 1,
         "history": 4096, "top_k": 40, "mixed": False},
        # a full serving batch, every row with its own history and parameters: the largest call
        {"name": "sample_64_rows", "kind": "sample", "vocab": FULL_V, "d": FULL_D, "rows": 64,
         "history": 2048, "top_k": 64, "mixed": True},
        # speculative decoding: four drafts verified greedily in one pass
        {"name": "verify_greedy_5_rows", "kind": "verify_greedy", "vocab": FULL_V, "d": FULL_D, "rows": 5,
         "norm": False},
        # the same from the residual stream, with the model's last norm in front, on a mid-sized
        # head and six drafts
        {"name": "verify_norm_7_rows", "kind": "verify_greedy", "vocab": 151669, "d": 3584, "rows": 7,
         "norm": True},
        # the decode loop as a program drives it: one request of 32 tokens, each read back
        {"name": "generate_32", "kind": "generate", "vocab": FULL_V, "d": FULL_D, "steps": 32,
         "prompt": 512, "top_k": 64},
        # selection over one row of logits that another library computed
        {"name": "select_1_row", "kind": "select", "vocab": FULL_V, "rows": 1, "top_k": 64},
        # a batch of such rows on an odd vocabulary, no top-k: rows that start at any alignment
        {"name": "select_48_rows", "kind": "select", "vocab": 151669, "rows": 48, "top_k": 0},
        # wide shortlists: diverse sampling with top_k in the thousands
        {"name": "select_wide_8_rows", "kind": "select", "vocab": FULL_V, "rows": 8, "top_k": 1000},
        # speculative sampling: four drafts with the draft model's logits, the rejection test
        {"name": "verify_draft_5_rows", "kind": "verify_draft", "vocab": FULL_V, "rows": 5},
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["greedy", "logits", "sample", "verify_greedy", "generate", "select", "select",
                       "verify_draft"])
    case = {"kind": kind, "vocab": _log_int(rng, 32000, FULL_V)}
    if kind in ("greedy", "logits", "sample", "verify_greedy", "generate"):
        case["d"] = 128 * _log_int(rng, 8, 42)
    if kind in ("greedy", "logits", "sample", "select"):
        case["rows"] = _log_int(rng, 1, 64)
    if kind == "sample":
        case["history"] = _log_int(rng, 16, 4096)
        case["mixed"] = rng.random() < 0.5
    if kind == "verify_greedy":
        case["norm"] = rng.random() < 0.5
        case["rows"] = rng.randint(2, 8 if case["norm"] else 9)
    if kind == "verify_draft":
        case["rows"] = rng.randint(2, 9)
    if kind == "generate":
        case["steps"] = rng.randint(8, 32)
        case["prompt"] = _log_int(rng, 16, 4000)
    if kind in ("sample", "generate", "select"):
        case["top_k"] = rng.choice([0, _log_int(rng, 1, 256), _log_int(rng, 10, 200),
                                    _log_int(rng, 257, 4096) if kind == "select" else 64])
    return case


# ---- inputs ---------------------------------------------------------------------------------------

def _gen(seed, stream):
    return torch.Generator(device=DEV).manual_seed((seed * 1000003 + stream) & 0x7FFFFFFFFFFFFFFF)


def _weights(case, seed):
    """The head's [W | S | B] slice: W u32 [V][d/8], nibble j of a word its column j; S, B bf16."""
    v, d = case["vocab"], case["d"]
    g = _gen(seed, 1)
    W = torch.empty(v, d // 8, dtype=torch.int32, device=DEV)
    S = torch.empty(v, d // GROUP, dtype=torch.bfloat16, device=DEV)
    B = torch.empty(v, d // GROUP, dtype=torch.bfloat16, device=DEV)
    shift = torch.arange(0, 32, 4, dtype=torch.int32, device=DEV)
    for r0 in range(0, v, 32768):
        n = min(32768, v - r0)
        w = torch.randn(n, d // GROUP, GROUP, generator=g, device=DEV) * (SIGMA * math.sqrt(168.0 / d))
        lo, hi = w.amin(2), w.amax(2)
        s, b = ((hi - lo) / 15.0).bfloat16(), lo.bfloat16()
        q = ((w - b.float()[..., None]) / s.float()[..., None]).round().clamp_(0, 15).to(torch.int32)
        W[r0:r0 + n] = (q.view(n, d // 8, 8) << shift).sum(2, dtype=torch.int64).to(torch.int32)
        S[r0:r0 + n], B[r0:r0 + n] = s, b
    return W, S, B


def _head(case, seed):
    W, S, B = _weights(case, seed)
    wsb = torch.cat([t.contiguous().view(torch.uint8).view(-1) for t in (W, S, B)])
    return twd.LMHead(wsb, case["vocab"], case["d"], CAP)


def _hidden(case, seed, rows):
    return torch.randn(rows, case["d"], generator=_gen(seed, 2), device=DEV).bfloat16()


def _residual(case, seed, rows):
    """The residual stream before the last norm, and the norm's weight."""
    g = _gen(seed, 2)
    x = 12.0 * torch.randn(rows, case["d"], generator=g, device=DEV)
    w = (1.0 + 0.25 * torch.randn(case["d"], generator=g, device=DEV)).bfloat16()
    return x, w


def _history(case, seed, rows):
    return torch.randint(0, case["vocab"], (rows * case["history"],), generator=_gen(seed, 3), device=DEV,
                         dtype=torch.int32)


def _params(case, seed, rows):
    """Per-row parameters: all alike, or every row its own."""
    r = np.random.default_rng(seed)
    n_hist = case.get("history", 0)
    out = []
    for m in range(rows):
        t, p, k, rp = 0.8, 0.95, case["top_k"], 1.1 if n_hist else 1.0
        if case.get("mixed"):
            t, p = float(r.uniform(0.5, 1.2)), float(r.uniform(0.8, 0.98))
            k = int(r.integers(1, 2 * k + 1)) if k else 0
        out.append(twd.RowParams(t, p, min(k, 256) if n_hist else k, rp, float(np.float32(r.uniform(0, 0.9999))),
                                 CAP if n_hist else 0.0, m * n_hist, n_hist))
    return out


def _logits(case, seed, rows):
    """Rows of softcapped logits, as another library's head writes them."""
    z = 3.6 * torch.randn(rows, case["vocab"], generator=_gen(seed, 4), device=DEV)
    return CAP * torch.tanh(z / CAP)


def prepare(case, seed):
    kind, st = case["kind"], dict(case)
    v = case["vocab"]
    if kind in ("greedy", "logits", "sample"):
        rows = case["rows"]
        st["head"] = _head(case, seed)
        st["hidden"] = _hidden(case, seed, rows)
        st["logits"] = torch.empty(rows, v, dtype=torch.float32, device=DEV)
        st["tokens"] = torch.empty(rows, dtype=torch.int32, device=DEV)
        if kind == "sample":
            st["params"], st["history_ids"] = _params(case, seed, rows), _history(case, seed, rows)
    elif kind == "verify_greedy":
        rows = case["rows"]
        st["head"] = _head(case, seed)
        if case["norm"]:
            st["x"], st["norm_w"] = _residual(case, seed, rows)
            best = st["head"].greedy_rmsnorm(st["x"], st["norm_w"], EPS)
        else:
            st["hidden"] = _hidden(case, seed, rows)
            best = st["head"].greedy(st["hidden"])
        # a draft model that is right with p = 0.7 per position
        g = _gen(seed, 5)
        other = torch.randint(0, v, (rows - 1,), generator=g, device=DEV, dtype=torch.int32)
        right = torch.rand(rows - 1, generator=g, device=DEV) < 0.7
        st["drafts"] = torch.where(right, best[:rows - 1], other)
        st["logits"] = torch.empty(rows, v, dtype=torch.float32, device=DEV)
        st["result"] = torch.zeros(twd.VERIFY_WORDS, dtype=torch.int32, device=DEV)
    elif kind == "generate":
        st["head"] = _head(case, seed)
        st["hidden"] = _hidden(case, seed, case["steps"])
        st["prompt_ids"] = [int(t) for t in np.random.default_rng(seed).integers(0, v, case["prompt"])]
        st["sampling"] = twd.SamplingParams(0.8, 0.95, case["top_k"], 1.1, True, seed)
    elif kind == "select":
        st["logits"] = _logits(case, seed, case["rows"])
        st["params"] = _params(case, seed, case["rows"])
        st["tokens"] = torch.empty(case["rows"], dtype=torch.int32, device=DEV)
        st["selector"] = twd.Selector(v, case["rows"])
    else:  # verify_draft: the draft model's logits lie near the target's, the drafts are its samples
        rows = case["rows"]
        st["logits"] = _logits(case, seed, rows)
        g = _gen(seed, 5)
        d = st["logits"][:rows - 1] + 0.5 * torch.randn(rows - 1, v, generator=g, device=DEV)
        st["draft_rows"] = [r.clone() for r in d]
        noise = -torch.log(-torch.log(torch.rand(rows - 1, v, generator=g, device=DEV).clamp_(1e-9, 1 - 1e-7)))
        st["drafts"] = (d / 0.8 + noise).argmax(1).to(torch.int32)
        st["params"] = twd.RowParams(0.8, 0.95, 64, 1.0, 0.0, CAP, 0, 0)
        st["seed"] = seed
        st["selector"] = twd.Selector(v, rows)
        st["result"] = torch.zeros(twd.VERIFY_WORDS, dtype=torch.int32, device=DEV)
    return st


def run(st):
    kind = st["kind"]
    if kind == "greedy":
        st["head"].greedy(st["hidden"], logits=st["logits"], tokens=st["tokens"])
        return {"logits": st["logits"], "tokens": st["tokens"]}
    if kind == "logits":
        return {"logits": st["head"].logits(st["hidden"], out=st["logits"])}
    if kind == "sample":
        st["head"].sample(st["hidden"], st["params"], history=st["history_ids"], logits=st["logits"],
                          tokens=st["tokens"])
        return {"logits": st["logits"], "tokens": st["tokens"]}
    if kind == "verify_greedy":
        if st["norm"]:
            st["head"].verify_greedy_rmsnorm(st["x"], st["norm_w"], st["drafts"], EPS, logits=st["logits"],
                                             result=st["result"])
        else:
            st["head"].verify_greedy(st["hidden"], st["drafts"], logits=st["logits"], result=st["result"])
        return {"logits": st["logits"], "result": st["result"]}
    if kind == "generate":
        gen = twd.Generator(st["head"], st["sampling"], st["prompt_ids"], st["steps"])
        for h in st["hidden"]:
            if gen.step(h)[1]:
                break
        ids = np.array(gen.tokens()[st["prompt"]:], dtype=np.int64)
        gen.close()
        return ids
    if kind == "select":
        return st["selector"].select(st["logits"], st["params"], tokens=st["tokens"])
    return st["selector"].verify_draft(st["logits"], st["draft_rows"], st["params"], st["seed"], st["drafts"],
                                       result=st["result"])


def work(case):
    """Bytes: the head's 4-bit weights with their scales and biases, hidden rows, histories and
    logits, each once. Flops: two per weight and row."""
    kind, v = case["kind"], case["vocab"]
    if kind == "select":
        return {"bytes": 4 * v * case["rows"] + 36 * case["rows"], "flops": 0}
    if kind == "verify_draft":
        return {"bytes": 4 * v * (2 * case["rows"] - 1) + 4 * twd.VERIFY_WORDS, "flops": 0}
    d = case["d"]
    weights = v * (d // 2 + d // GROUP * 4)
    if kind == "generate":  # one logit row a step stays with the loop
        n = case["steps"]
        return {"bytes": n * (weights + 2 * d + 4 * (case["prompt"] + n // 2)), "flops": 2 * v * d * n}
    rows = case["rows"]
    n = weights + (4 if case.get("norm") else 2) * d * rows + 4 * v * rows
    n += 4 * case.get("history", 0) * rows
    return {"bytes": n, "flops": 2 * v * d * rows}


def tolerance(case):
    # Selection over given logits is exact: the same ids, whatever the order of its sums. Logits are
    # fp32 sums of exact products, 2e-6 to 8e-6 (2-norm) from the 64-bit ones in the orders measured;
    # an id drawn from them changes only where a cut or a draw falls within that rounding.
    if case["kind"] in ("select", "verify_draft"):
        return "exact"
    return {"rel": 3e-5, "max": 3e-4, "differ": 0.01}


# ---- the same in 64 bits, in plain torch ------------------------------------------------------------

def _exact_logits(case, seed):
    W, S, B = _weights(case, seed)
    v, d, rows = case["vocab"], case["d"], case["rows"]
    if case.get("norm"):
        x, w = _residual(case, seed, rows)
        x = x.double()
        h = x / torch.sqrt(x.square().mean(1, keepdim=True) + EPS) * w.double()
    else:
        h = _hidden(case, seed, rows).double()
    shift = torch.arange(0, 32, 4, dtype=torch.int32, device=DEV)
    out = torch.empty(rows, v, dtype=torch.float64, device=DEV)
    for r0 in range(0, v, 16384):
        n = min(16384, v - r0)
        q = ((W[r0:r0 + n, :, None] >> shift) & 15).view(n, d // GROUP, GROUP)
        w = q.double() * S[r0:r0 + n].double()[..., None] + B[r0:r0 + n].double()[..., None]
        out[:, r0:r0 + n] = torch.mm(h, w.view(n, d).t().contiguous())
    return CAP * torch.tanh(out / CAP)


def exact(case, seed):
    kind = case["kind"]
    if kind not in ("greedy", "logits", "sample", "verify_greedy"):
        return None
    logits = _exact_logits(case, seed)
    if kind == "logits":
        return {"logits": logits}
    if kind == "verify_greedy":
        return {"logits": logits, "result": None}
    if kind == "sample":
        # each occurrence of an id in the row's history divides or multiplies its logit once more
        ids, params = _history(case, seed, case["rows"]).long(), _params(case, seed, case["rows"])
        for m, p in enumerate(params):
            count = torch.bincount(ids[p.history_offset:p.history_offset + p.history_len], minlength=case["vocab"])
            rp, lim = float(np.float32(p.repetition_penalty)), float(np.float32(CAP) * np.float32(0.9999))
            for n in range(1, int(count.max()) + 1):
                x = logits[m]
                y = torch.where(x > 0, x / rp, x * rp).clamp(-lim, lim)
                logits[m] = torch.where(count >= n, y, x)
    return {"logits": logits, "tokens": None}
