"""The calls this library is used for, as cases that can be timed: what a serving engine asks of its token sampler, from a
lone decode row to a full masked batch, through the public entry points of the package.

Inputs are drawn on the GPU from the case's seed. Logits are synthetic (normal, Zipfian, or normal with a few raised tokens,
which is what a confident model's rows look like), histories lean towards low token ids and have another length on every
row, and a batch tells the sampler what is known about its rows (no top-k at all, a bound on it, a min-p on the rows without
one) by the same rule whirl-llm_amd/workloads.py follows.

Results compared are the sampler's answers: tokens, their probabilities, kept counts, row maxima and normalisers, lists,
acceptance counts. The sampler's diagnostic words (the route bits in its flags, the distances to the nearest decision) say
how an implementation got there and are not among them."""
import math

import torch

from __graft_entry__ import load_package

ws = load_package()
DEV = "cuda:0"

# Vocabularies: 151936, 262144, 50257 and 32000 are the ones of this repository's workloads and tests.
LISTED = [
    # one user decoding: the latency of a single row under the reference's usual settings
    dict(name="decode_1_top_k", path="sample", rows=1, vocab=151936, dtype="f32", logits="raised", sigma=2.0, temp_lo=0.8, temp_hi=0.8, filters="top_k",
         top_k=40, top_p_lo=0.95, top_p_hi=0.95, min_p=0.0, hist=256, bias=0, allowed=1.0),
    # a busy server: every request with settings of its own, penalties over long texts, logit bias
    dict(name="batch_64_mixed", path="sample", rows=64, vocab=151936, dtype="f32", logits="normal", sigma=2.0, temp_lo=0.5, temp_hi=1.2, filters="mixed",
         top_k=50, top_p_lo=0.8, top_p_hi=1.0, min_p=0.05, hist=4096, bias=300, allowed=1.0),
    # a full decode batch with top-p alone, penalties on: the select over the whole vocabulary
    dict(name="batch_256_top_p", path="sample", rows=256, vocab=151936, dtype="f32", logits="normal", sigma=2.0, temp_lo=0.7, temp_hi=1.0, filters="top_p",
         top_k=0, top_p_lo=0.9, top_p_hi=0.9, min_p=0.0, hist=2048, bias=0, allowed=1.0),
    # the same from a model that leaves its logits in bf16: half the bytes, hundreds of equal logits at the cut
    dict(name="batch_256_bf16_top_p", path="sample", rows=256, vocab=151936, dtype="bf16", logits="zipf", sigma=0.3, temp_lo=1.0, temp_hi=1.0,
         filters="top_p", top_k=0, top_p_lo=0.9, top_p_hi=0.9, min_p=0.0, hist=2048, bias=0, allowed=1.0),
    # requests that set top-k or leave it out, with the usual range of top-p, on bf16 logits: a batch of which nothing is known
    dict(name="batch_64_bf16_any", path="sample", rows=64, vocab=151936, dtype="bf16", logits="raised", sigma=2.0, temp_lo=0.6, temp_hi=1.2, filters="mixed",
         top_k=50, top_p_lo=0.8, top_p_hi=0.99, min_p=0.0, hist=1024, bias=0, allowed=1.0),
    # constrained decoding at full size: nine tokens in ten masked out, long texts, a wide top-k. The largest case
    dict(name="batch_1024_masked", path="sample", rows=1024, vocab=262144, dtype="f32", logits="normal", sigma=3.0, temp_lo=1.0, temp_hi=1.0, filters="top_k",
         top_k=1000, top_p_lo=0.95, top_p_hi=0.95, min_p=0.0, hist=8192, bias=500, allowed=0.1),
    # a vocabulary of odd size, so that most rows start off any vector boundary
    dict(name="batch_32_odd_vocab", path="sample", rows=32, vocab=50257, dtype="f32", logits="normal", sigma=2.0, temp_lo=0.7, temp_hi=1.0, filters="mixed",
         top_k=50, top_p_lo=0.8, top_p_hi=1.0, min_p=0.05, hist=500, bias=20, allowed=1.0),
    # greedy decoding of a batch
    dict(name="greedy_32", path="greedy", rows=32, vocab=151936),
    # the engine's candidate lists for its host-side filter, a decode batch of eight
    dict(name="candidates_8", path="candidates", rows=8, vocab=151936, k=256),
    # classic speculative verification
    dict(name="verify_32x9", path="verify", rows=32, positions=9, vocab=151936),
    # one cycle of sampled speculative decoding: drafts position by position, then every verify row in one launch, then acceptance
    dict(name="cycle_8x4", path="cycle", rows=8, drafts=4, vocab=151936, top_k=40, hist=512),
    # a request decoded through the C++ host API, token by token
    dict(name="host_decode_32", path="host_decode", rows=1, steps=32, vocab=151936, top_k=40, hist=256),
]


def listed():
    return [dict(c) for c in LISTED]


def _log_int(rng, lo, hi):
    return max(lo, min(hi, int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))))


def _vocab(rng, lo=8000, hi=262144):
    """Half the vocabularies are padded to a multiple of 64, as most models' are; the others are whatever they are."""
    v = _log_int(rng, lo, hi)
    return v // 64 * 64 if rng.random() < 0.5 else v


def draw(rng):
    path = rng.choices(["sample", "greedy", "candidates", "verify", "cycle", "host_decode"], [8, 1, 1, 1, 1, 1])[0]
    vocab = _vocab(rng)
    if path == "greedy":
        return dict(path=path, rows=_log_int(rng, 1, 256), vocab=vocab)
    if path == "candidates":
        return dict(path=path, rows=_log_int(rng, 1, 32), vocab=_vocab(rng, 32000), k=rng.choice([4, 64, 256, 16384]))
    if path == "verify":
        return dict(path=path, rows=_log_int(rng, 1, 64), positions=rng.randint(2, 9), vocab=vocab)
    if path == "cycle":
        return dict(path=path, rows=rng.randint(1, 16), drafts=rng.randint(1, 7), vocab=vocab, top_k=rng.choice([20, 40, 50]), hist=_log_int(rng, 16, 2048))
    if path == "host_decode":
        return dict(path=path, rows=1, steps=rng.randint(8, 64), vocab=vocab, top_k=rng.choice([20, 40, 50]), hist=_log_int(rng, 16, 2048))
    dtype = rng.choice(["f32", "bf16"])
    rows = _log_int(rng, 1, min(1024, max(1, 400_000_000 // (vocab * 4))))
    filters = rng.choice(["top_k", "mixed", "mixed", "top_p", "top_p", "min_p"])
    logits = rng.choice(["normal", "raised", "raised", "zipf"])
    lo = rng.uniform(0.6, 1.0)
    p = rng.uniform(0.8, 0.95)
    return dict(path=path, rows=rows, vocab=vocab, dtype=dtype, logits=logits, sigma=round(rng.uniform(0.2, 0.5) if logits == "zipf" else rng.uniform(1.5, 3.0), 2),
                temp_lo=round(lo, 2), temp_hi=round(lo + rng.uniform(0.0, 0.4), 2), filters=filters,
                top_k=0 if filters in ("top_p", "min_p") else _log_int(rng, 1, 1000) if filters == "top_k" else 50,
                top_p_lo=round(p, 3), top_p_hi=round(p + rng.uniform(0.0, 0.04), 3),
                min_p=round(rng.uniform(0.02, 0.1), 3) if filters == "min_p" or (filters == "mixed" and rng.random() < 0.5) else 0.0,
                hist=rng.choice([0, _log_int(rng, 16, 4096)]), bias=rng.choice([0, 0, _log_int(rng, 4, 300)]),
                allowed=rng.choice([1.0, 1.0, 1.0, round(rng.uniform(0.1, 0.9), 2)]))


# ---- inputs ---------------------------------------------------------------------------------------------------------

def _logits(g, rows, vocab, kind, sigma):
    """[rows, vocab] fp32. normal: N(0, sigma). raised: the same with 2 to 40 tokens a row lifted to 10 .. 14. zipf: -1.1 ln(rank)
    over a random order of the vocabulary, plus N(0, sigma)."""
    x = torch.empty((rows, vocab), device=DEV).normal_(0.0, sigma, generator=g)
    if kind == "zipf":
        base = -1.1 * torch.log(torch.arange(1, vocab + 1, device=DEV, dtype=torch.float32))
        for r in range(0, rows, 64):  # (in slices: the random orders take eight bytes a token)
            order = torch.rand((min(64, rows - r), vocab), device=DEV, generator=g).argsort(dim=1)
            x[r:r + 64] += base[order]
    elif kind == "raised":
        top = torch.empty((rows, 40), device=DEV).uniform_(10.0, 14.0, generator=g)
        ids = torch.randint(0, vocab, (rows, 40), device=DEV, generator=g)
        n = torch.randint(2, 41, (rows, 1), device=DEV, generator=g)
        lifted = torch.where(torch.arange(40, device=DEV) < n, top, x.gather(1, ids))
        x.scatter_reduce_(1, ids, lifted, "amax")  # (the larger of two that fall on one token)
    return x


def _ids(g, n, vocab):
    """Token ids of a text: low ids, the frequent ones of a vocabulary, come up more often."""
    return (torch.rand(n, device=DEV, generator=g).square() * vocab).to(torch.int32).clamp_(0, vocab - 1)


def _lists(g, rows, most):
    """Offsets of `rows` lists of another length each, from a quarter of `most` up to it, and their total."""
    n = torch.randint(max(1, most // 4), most + 1, (rows,), device=DEV, generator=g, dtype=torch.int64)
    off = torch.zeros(rows + 1, dtype=torch.int32, device=DEV)
    off[1:] = n.cumsum(0).to(torch.int32)
    return off, int(off[-1])


def _bitmap(g, rows, vocab, share):
    """Allow bitmap, [rows, ceil(vocab / 32)] words."""
    words = (vocab + 31) // 32
    bit = torch.tensor([1 << i if i < 31 else -(1 << 31) for i in range(32)], dtype=torch.int32, device=DEV)
    out = torch.empty((rows, words), dtype=torch.int32, device=DEV)
    for r in range(0, rows, 64):
        on = torch.rand((min(64, rows - r), words, 32), device=DEV, generator=g) < share
        out[r:r + 64] = torch.where(on, bit, 0).sum(2, dtype=torch.int32)
    return out


def _sampler(g, c):
    rows, vocab = c["rows"], c["vocab"]
    x = _logits(g, rows, vocab, c["logits"], c["sigma"])
    if c["dtype"] == "bf16":
        x = x.to(torch.bfloat16)

    def uniform(lo, hi, dt=torch.float64):
        return (torch.rand(rows, device=DEV, generator=g, dtype=torch.float64) * (hi - lo) + lo).to(dt)

    args = dict(inv_t=uniform(c["temp_lo"], c["temp_hi"]).reciprocal().to(torch.float32), top_p=uniform(c["top_p_lo"], c["top_p_hi"]),
                min_p=torch.full((rows,), c["min_p"], dtype=torch.float64, device=DEV),
                seed=torch.randint(0, 1 << 62, (rows,), device=DEV, generator=g), step=torch.randint(0, 5000, (rows,), device=DEV, generator=g))
    if c["filters"] == "top_k":
        args.update(top_k=torch.full((rows,), c["top_k"], dtype=torch.int32, device=DEV), top_k_max=c["top_k"])
    elif c["filters"] == "mixed":  # no top-k, 20, or the case's: bounded only where the rows without one have a min-p
        pick = torch.tensor([0, 20, c["top_k"]], dtype=torch.int32, device=DEV)
        args.update(top_k=pick[torch.randint(0, 3, (rows,), device=DEV, generator=g)])
        if c["min_p"] >= 1e-3:
            args.update(top_k_max=c["top_k"], min_p_min=c["min_p"])
    elif c["filters"] == "min_p":
        args.update(min_p_min=c["min_p"])
    if c["hist"]:
        off, total = _lists(g, rows, c["hist"])
        args.update(hist=_ids(g, total, vocab), hist_off=off, max_hist=c["hist"])
        args.update({k: torch.full((rows,), v, device=DEV) for k, v in (("rep", 1.1), ("pres", 0.3), ("freq", 0.02))})
    if c["bias"]:
        off, total = _lists(g, rows, c["bias"])
        args.update(bias_ids=torch.randint(0, vocab, (total,), device=DEV, generator=g, dtype=torch.int32),
                    bias_vals=torch.empty(total, device=DEV).uniform_(-5.0, 5.0, generator=g), bias_off=off, max_bias=c["bias"])
    if c["allowed"] < 1.0:
        args.update(allow=_bitmap(g, rows, vocab, c["allowed"]))
    return ws.BatchSampler(x, args.pop("inv_t"), args.pop("seed"), args.pop("step"), rng=ws.RNG_PHILOX, want_margin=False, **args)


def _workspace(nbytes):
    return torch.zeros(nbytes, dtype=torch.uint8, device=DEV) if nbytes else None


def _verify(g, c):
    n, pos, vocab = c["rows"], c["positions"], c["vocab"]
    t = _logits(g, n * pos, vocab, "normal", 2.0)
    d = 0.7 * t + 0.3 * _logits(g, n * pos, vocab, "normal", 2.0)
    p, q = (torch.softmax(v, -1).reshape(n, pos, vocab) for v in (t, d))
    cum = q[:, :-1].reshape(-1, vocab).cumsum(1)
    u = torch.rand((cum.shape[0], 1), device=DEV, generator=g) * cum[:, -1:]
    draft = torch.searchsorted(cum, u).clamp_(max=vocab - 1).reshape(n, pos - 1).to(torch.int32)
    s = dict(p=p, q=q, draft=draft, seed=torch.randint(0, 1 << 62, (n,), device=DEV, generator=g), step0=torch.randint(0, 5000, (n,), device=DEV, generator=g))
    shape = ws.SpecVerify(p.data_ptr(), q.data_ptr(), draft.data_ptr(), n, pos, vocab)
    s["workspace"] = _workspace(int(ws.lib().ws_spec_verify_workspace(ws.C.byref(shape))))
    return s


def _cycle(g, c):
    n, nd, vocab = c["rows"], c["drafts"], c["vocab"]
    x = _logits(g, n * (nd + 1), vocab, "raised", 2.0).reshape(n, nd + 1, vocab)
    # the draft head sees nearly what the model will see, position by position
    heads = [(x[:, j] + torch.empty((n, vocab), device=DEV).normal_(0.0, 0.5, generator=g)).contiguous() for j in range(nd)]
    cap = c["hist"] + nd + 2
    H = ws.DeviceHistory(n, cap, DEV)
    H.tokens.copy_(_ids(g, n * cap, vocab).reshape(n, cap))
    H.len.copy_(torch.randint(max(1, c["hist"] // 4), c["hist"] + 1, (n,), device=DEV, generator=g))
    H.n_gen.copy_(torch.randint(0, 5000, (n,), device=DEV, generator=g))
    rows = n * (nd + 1)
    i32 = dict(dtype=torch.int32, device=DEV)
    ctl = torch.zeros((n, ws.CTL_WORDS), **i32)
    ctl[:, 48] = nd
    s = dict(heads=heads, hist=H, slot=torch.arange(n, **i32), ctl=ctl, area_host=[i * ws.CTL_WORDS for i in range(n)],
             area=torch.arange(n, **i32) * ws.CTL_WORDS, row0=torch.arange(n, **i32) * (nd + 1), hist_off=torch.zeros(rows, **i32),
             hist_len=torch.zeros(rows, **i32), query=torch.zeros(rows, **i32), step=torch.zeros(rows, dtype=torch.int64, device=DEV),
             qbuf=torch.zeros(n * ws.Q_WORDS, **i32), workspace=_workspace(int(ws.lib().ws_draft_sample_rows_workspace(vocab, n))))
    keys = torch.randint(0, 1 << 62, (nd, n), device=DEV, generator=g).tolist()
    s["draft_args"] = [[dict(top_k=20, qoff=i * ws.Q_WORDS, inv_t=1.25, top_p=0.95, min_p=0.02, key=keys[j][i]) for i in range(n)] for j in range(nd)]

    def full(v, dt):
        return torch.full((rows,), v, dtype=dt, device=DEV)

    seed = torch.randint(0, 1 << 62, (n, 1), device=DEV, generator=g).expand(n, nd + 1).reshape(-1).contiguous()
    s["sampler"] = ws.BatchSampler(x.reshape(rows, vocab), full(1.25, torch.float32), seed, s["step"], top_k=full(c["top_k"], torch.int32),
                                   top_p=full(0.95, torch.float64), rng=ws.RNG_SPLITMIX, hist=H.tokens.reshape(-1), hist_off=s["hist_off"],
                                   hist_len=s["hist_len"], max_hist=cap, rep=full(1.1, torch.float32), pres=full(0.3, torch.float32),
                                   freq=full(0.02, torch.float32), query=s["query"], want_entropy=True, want_margin=False, top_k_max=c["top_k"])
    # where the answers stand: drafts and kept tokens in the control areas, the draft distributions in qbuf
    s["answers"] = dict(drafts=ctl[:, 16:16 + nd], kept=ctl[:, :nd + 1], q=s["qbuf"].view(torch.float32).reshape(n, ws.Q_WORDS)[:, 33:65])
    return s


def prepare(case, seed):
    g = torch.Generator(device=DEV).manual_seed(seed)
    path, rows, vocab = case["path"], case["rows"], case["vocab"]
    if path == "sample":
        return dict(path=path, sampler=_sampler(g, case))
    if path == "verify":
        return dict(path=path, **_verify(g, case))
    if path == "cycle":
        return dict(path=path, **_cycle(g, case))
    x = _logits(g, rows, vocab, "raised", 2.0)
    if path == "greedy":
        return dict(path=path, x=x)
    if path == "candidates":
        return dict(path=path, x=x, k=case["k"], workspace=ws.topk_rows_workspace(vocab, case["k"], rows, DEV))
    return dict(path=path, row=x[0], top_k=case["top_k"], steps=case["steps"], hist=_ids(g, case["hist"], vocab).cpu().numpy(), seed=seed)


# ---- one pass -------------------------------------------------------------------------------------------------------

def run(s):
    path = s["path"]
    if path == "sample":
        b = s["sampler"].run()
        return dict(token=b.token, prob=b.prob, n_kept=b.n_kept, stats=b.stats)
    if path == "greedy":
        return ws.argmax_rows(s["x"])
    if path == "candidates":
        return ws.topk_rows(s["x"], s["k"], 1.25, s["workspace"])
    if path == "verify":
        n_accepted, tokens, _ = ws.spec_verify_classic(s["p"], s["q"], s["draft"], s["seed"], s["step0"], workspace=s["workspace"], split=s["workspace"] is not None)
        return n_accepted, tokens
    if path == "cycle":
        for r, (head, args) in enumerate(zip(s["heads"], s["draft_args"])):
            ws.draft_sample_rows(head, s["ctl"], s["area_host"], r, args, s["qbuf"], workspace=s["workspace"])
        ws.history_stage(s["hist"], s["slot"], s["ctl"], s["area"], s["row0"], s["hist_off"], s["hist_len"], s["query"], s["step"])
        b = s["sampler"].run()
        typical = dict(query_prob=b.query_prob, entropy=b.entropy, eps=0.09, delta=0.3)
        n_accepted, chosen, _, relaxed = ws.accept_sampled(b.token, b.flags, s["row0"], s["ctl"], s["area"], typical=typical)
        return dict(s["answers"], n_accepted=n_accepted, chosen=chosen, relaxed=relaxed, token=b.token, prob=b.prob, n_kept=b.n_kept,
                    query_prob=b.query_prob, entropy=b.entropy)
    tokens, _, n_kept, _ = ws.host_decode_steps(s["row"], 1.25, s["seed"], 0, s["steps"], top_k=s["top_k"], top_p=0.95, hist=s["hist"], rep=1.1)
    return tokens, int(n_kept)


# ---- what a pass cannot do without ----------------------------------------------------------------------------------

def work(case):
    """Bytes: every logit once, the penalty lists (their lengths on average five eighths of the most), the bitmap, the results.
    Operations: two per logit where a row's normaliser is wanted (scale, sum), one where only its order is."""
    path, rows, vocab = case["path"], case["rows"], case["vocab"]
    if path == "sample":
        each = 2 if case["dtype"] == "bf16" else 4
        lists = 0.625 * (4 * case["hist"] + 8 * case["bias"])
        return {"bytes": rows * (vocab * each + lists + (vocab / 8 if case["allowed"] < 1.0 else 0) + 60 + 20), "flops": 2 * rows * vocab}
    if path == "greedy":
        return {"bytes": rows * (vocab * 4 + 4), "flops": rows * vocab}
    if path == "candidates":
        return {"bytes": rows * (vocab * 4 + case["k"] * 8 + 8), "flops": 2 * rows * vocab}
    if path == "verify":  # two probabilities a draft, and one pair of rows a sequence for the token after the last accepted one
        return {"bytes": rows * (8 * (case["positions"] - 1) + 8 * vocab + 4 * case["positions"] + 20), "flops": 2 * rows * vocab}
    if path == "cycle":
        n = rows * (2 * case["drafts"] + 1)
        return {"bytes": n * (vocab * 4 + 80) + rows * 4 * case["hist"], "flops": 2 * n * vocab}
    return {"bytes": case["steps"] * (vocab * 4 + case["hist"] * 4 + 40), "flops": 2 * case["steps"] * vocab}


def tolerance(case):
    """Tokens and counts are exact, but for the few rows whose cut or draw lies within the rounding of a 32-bit normaliser of a
    token's edge. Probabilities and normalisers are 32-bit sums over the row."""
    if case["path"] == "greedy":
        return "exact"
    return {"rel": 1e-5, "differ": 0.01}
