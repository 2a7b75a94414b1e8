"""The work a serving program has the token sampler do, as measurable cases.

Each case is one pass through the package's entry points (`Sampler` and its
pre-built launchers), over inputs made on the GPU from a seed:

  pick     one batched pick: penalties, bias, mask, top-k, top-p, min-p and the
           inverse-CDF draw, or greedy
  race     the same kept set with the race-v2 winner instead of the draw
  step     an engine step: every row's pick and its log-probability receipt
  topn     the full-vocabulary log-softmax with its n most likely IDs
  spec     speculative verification of drafted tokens
  lm_head  the bf16 lm_head GEMM with tile statistics and the pick from them

`exact` restates each of them in plain torch in 64 bits.
"""
from __future__ import annotations

import math

import torch

from metallix_amd import Sampler

QWEN3_VOCAB = 151936
GEMMA_VOCAB = 262144
OUT_BYTES = 4 + 8 + 4 + 4          # token, sampling_logprob, status, kept_count
MAX_BYTES = 256 * GEMMA_VOCAB * 4  # the largest logit batch a drawn case takes

# A pick case's logits:
#   "normal"  N(0, spread^2) with `peaks` tokens raised by 4 to 10 (the shape
#             of the repository's benchmark batches)
#   "text"    the head a language model gives: N(0, 2.5^2), and 4096 tokens
#             whose logits fall from about 20 as a * ln(rank), a drawn per row
#             (probability ~ rank^-a)
# and its rules, one per row:
#   "greedy", "chat" (T .7, top_k 20, top_p .8), "mix" (top_k {0, 20, 50,
#   1000}, top_p, min_p .05), "nucleus" (top_p alone), "plain" (temperature
#   alone), "topk" (T 1, top_k 64, top_p .95), "minp" (min_p alone)
RULES = ("greedy", "chat", "mix", "nucleus", "plain", "topk", "minp")


def listed():
    return [
        # One interactive stream, greedy (evaluation and tool-call runs).
        dict(name="greedy_one", kind="pick", rows=1, vocab=QWEN3_VOCAB, dtype="f32", logits="normal", rule="greedy",
             history=0, bias=0, mask=False),
        # One interactive chat stream with Qwen3's recommended rule and a repetition penalty.
        dict(name="chat_one", kind="pick", rows=1, vocab=QWEN3_VOCAB, dtype="f32", logits="normal", rule="chat",
             history=512, bias=0, mask=False),
        # A serving batch in which every request brings its own rule and penalties: the headline batch.
        dict(name="serve_mix", kind="pick", rows=64, vocab=QWEN3_VOCAB, dtype="f32", logits="normal", rule="mix",
             history=2048, bias=0, mask=False),
        # Nucleus sampling without a top-k, the usual rule of an API request that sets top_p only.
        dict(name="nucleus", kind="pick", rows=32, vocab=QWEN3_VOCAB, dtype="f32", logits="text", rule="nucleus",
             history=0, bias=0, mask=False),
        # The API's default rule (temperature alone) with presence and frequency penalties and a
        # logit_bias list that raises and bans tokens; bf16 logits, a ragged batch and vocabulary.
        dict(name="api_default", kind="pick", rows=37, vocab=50257, dtype="bf16", logits="text", rule="plain",
             history=700, bias=24, mask=False),
        # Constrained decoding: bf16 logits under grammar masks, top_p alone.
        dict(name="grammar", kind="pick", rows=32, vocab=QWEN3_VOCAB, dtype="bf16", logits="normal", rule="nucleus",
             history=0, bias=0, mask=True),
        # The largest batch: 256 rows of a 262144-token vocabulary, top-k and top-p.
        dict(name="gemma_topk", kind="pick", rows=256, vocab=GEMMA_VOCAB, dtype="f32", logits="normal", rule="topk",
             history=0, bias=0, mask=False),
        # logprobs: the log-softmax head (the top 20 and 8 spares) of every row of that batch.
        dict(name="logprobs", kind="topn", rows=256, vocab=GEMMA_VOCAB, dtype="f32", n=28),
        # An engine step of the serving batch whose requests all ask for top_logprobs, two tokens suppressed.
        dict(name="engine_step", kind="step", rows=64, vocab=QWEN3_VOCAB, dtype="f32", logits="normal", rule="mix",
             history=2048, bias=0, mask=False, n=28, suppress=2),
        # Reproducible (race-v2) picks: half the rows under the serving rules, half over their whole row.
        dict(name="race", kind="race", rows=64, vocab=QWEN3_VOCAB, dtype="f32", logits="normal", rule="mix",
             history=2048, bias=0, mask=False, whole=2),
        # Speculative decoding: 16 sequences, 4 drafted tokens each.
        dict(name="spec_verify", kind="spec", rows=16, draft=4, vocab=QWEN3_VOCAB),
        # The head of a model: the bf16 lm_head of 64 rows with the pick fused into its epilogue.
        dict(name="lm_head", kind="lm_head", rows=64, hidden=1024, vocab=QWEN3_VOCAB),
    ]


def _log_int(rng, lo, hi):
    return int(round(math.exp(rng.uniform(math.log(lo), math.log(hi)))))


def draw(rng):
    kind = rng.choice(["pick"] * 6 + ["step", "race", "topn", "topn", "spec", "lm_head"])
    if kind == "spec":
        k = rng.randint(1, 8)
        vocab = _log_int(rng, 2000, QWEN3_VOCAB)
        rows = min(_log_int(rng, 1, 64), max(1, MAX_BYTES // (4 * (2 * k + 1) * vocab)))
        return dict(kind=kind, rows=rows, draft=k, vocab=vocab)
    if kind == "lm_head":
        hidden = 128 * _log_int(rng, 1, 32)
        vocab = 4 * _log_int(rng, 2000, GEMMA_VOCAB // 4)
        vocab = min(vocab, (QWEN3_VOCAB * 1024 // hidden) & ~3)
        return dict(kind=kind, rows=_log_int(rng, 1, 64), hidden=hidden, vocab=vocab)
    dtype = rng.choice(["f32", "bf16"])
    vocab = rng.choice([QWEN3_VOCAB, _log_int(rng, 2000, GEMMA_VOCAB), _log_int(rng, 20000, GEMMA_VOCAB)])
    rows = min(_log_int(rng, 1, 256), max(1, MAX_BYTES // (4 * vocab)))
    if kind == "topn":
        return dict(kind=kind, rows=rows, vocab=vocab, dtype=dtype, n=rng.choice([1, 8, 13, 28, 64]))
    rule = rng.choice(RULES)
    case = dict(kind=kind, rows=rows, vocab=vocab, dtype=dtype, logits=rng.choice(["normal", "text"]), rule=rule,
                history=rng.choice([0, _log_int(rng, 16, 8192)]), bias=rng.choice([0, 0, 0, _log_int(rng, 1, 300)]),
                mask=rng.random() < 0.25)
    if kind == "step":
        case.update(n=rng.choice([9, 13, 28]), suppress=rng.choice([0, 2, 5]), mask=False)
    if kind == "race":
        case.update(whole=rng.choice([0, 1, 2, 4]))
    return case


# ---------------------------------------------------------------------------
# Inputs

def _gen(seed):
    g = torch.Generator(device="cuda")
    g.manual_seed((int(seed) * 2654435761 + 12345) % (1 << 62))
    return g


def _uniform(g, shape, lo=0.0, hi=1.0):
    return lo + (hi - lo) * torch.rand(shape, generator=g, device="cuda", dtype=torch.float64)


def _logits(g, case, spread):
    """Logits [rows, stride], stride the vocabulary rounded up to 4."""
    R, V = case["rows"], case["vocab"]
    x = torch.zeros((R, (V + 3) // 4 * 4), dtype=torch.float32, device="cuda")
    x[:, :V] = spread * torch.randn((R, V), generator=g, device="cuda")
    rows = torch.arange(R, device="cuda")[:, None]
    if case.get("logits") == "text":
        H = min(4096, V // 2)
        ids = torch.randint(V, (R, H), generator=g, device="cuda")
        top = 20.0 + 2.0 * torch.randn((R, 1), generator=g, device="cuda")
        fall = _uniform(g, (R, 1), 1.2, 4.0).float()
        ln = torch.log(torch.arange(1, H + 1, device="cuda").float())[None, :]
        head = top - fall * ln + 0.3 * torch.randn((R, H), generator=g, device="cuda")
        x.scatter_reduce_(1, ids, head, "amax")
    else:
        n = 100 if spread > 2.9 else 50
        count = torch.randint(1, n + 1, (R, 1), generator=g, device="cuda")
        ids = torch.randint(V, (R, n), generator=g, device="cuda")
        amp = _uniform(g, (R, n), 4.0, 10.0).float() * (torch.arange(n, device="cuda")[None, :] < count)
        x.index_put_((rows.expand(R, n), ids), amp, accumulate=True)
    return x.to(torch.bfloat16) if case["dtype"] == "bf16" else x


def _zipf_ids(g, R, n, V):
    """n Zipf(1.1) ranks per row, mapped to IDs by one permutation."""
    w = torch.arange(1, V + 1, device="cuda", dtype=torch.float64) ** -1.1
    cdf = torch.cumsum(w, 0) / w.sum()
    perm = torch.randperm(V, generator=g, device="cuda")
    return perm[torch.searchsorted(cdf, _uniform(g, (R, n))).clamp_(max=V - 1)]


def _mask_words(g, R, V):
    """Grammar masks: runs of 1 to 64 legal tokens, 0.5 to 5% of the
    vocabulary; every ninth row allows exactly one token."""
    n = max(1, int(0.05 * V / 32.5))
    keep = (torch.arange(n, device="cuda")[None, :] < (_uniform(g, (R, 1), 0.1, 1.0) * n).clamp_(min=1.0))
    start = torch.randint(V, (R, n), generator=g, device="cuda")
    stop = torch.minimum(start + torch.randint(1, 65, (R, n), generator=g, device="cuda"), torch.tensor(V, device="cuda"))
    edge = torch.zeros((R, V + 1), dtype=torch.int32, device="cuda")
    edge.scatter_add_(1, start, keep.int())
    edge.scatter_add_(1, stop, -keep.int())
    legal = torch.cumsum(edge, 1)[:, :V] > 0
    legal[::9] = False
    legal[::9].scatter_(1, start[::9, :1], True)
    words = (V + 31) // 32
    bits = torch.zeros((R, words * 32), dtype=torch.int64, device="cuda")
    bits[:, :V] = legal
    w = (bits.view(R, words, 32) << torch.arange(32, device="cuda")).sum(2)
    return _i32(w)


def _i32(t):
    """int64 values below 2^32 as int32 bit patterns."""
    return torch.where(t >= 1 << 31, t - (1 << 32), t).to(torch.int32)


def _rules(g, case):
    """Per-row rule tensors of a pick (the keywords of Sampler.sample)."""
    R, rule = case["rows"], case["rule"]
    row = torch.arange(R, device="cuda")
    f64 = lambda v: torch.full((R,), float(v), dtype=torch.float64, device="cuda")
    kw = dict(temperature=f64(1.0), uniform=_uniform(g, (R,)))
    if rule == "greedy":
        kw["temperature"] = f64(0.0)
    elif rule == "chat":
        kw.update(temperature=f64(0.7), top_k=torch.full((R,), 20, dtype=torch.int32, device="cuda"), top_p=f64(0.8))
    elif rule == "mix":
        kw.update(temperature=_uniform(g, (R,), 0.3, 1.5), top_p=_uniform(g, (R,), 0.5, 1.0), min_p=f64(0.05),
                  top_k=torch.tensor([0, 20, 50, 1000], dtype=torch.int32, device="cuda")[row % 4])
    elif rule == "nucleus":
        kw["top_p"] = f64(0.95) if case["mask"] else _uniform(g, (R,), 0.8, 0.98)
        if not case["mask"]:
            kw["temperature"] = _uniform(g, (R,), 0.6, 1.0)
    elif rule == "plain":
        kw["temperature"] = _uniform(g, (R,), 0.7, 1.3)
    elif rule == "topk":
        kw.update(top_k=torch.full((R,), 64, dtype=torch.int32, device="cuda"), top_p=f64(0.95))
    elif rule == "minp":
        kw.update(temperature=_uniform(g, (R,), 0.7, 1.5), min_p=_uniform(g, (R,), 0.02, 0.2))
    return kw


def _lists(g, case, kw):
    """History, bias and mask tensors into kw."""
    R, V = case["rows"], case["vocab"]
    f32 = lambda v: torch.full((R,), float(v), dtype=torch.float32, device="cuda")
    if case["history"]:
        n = case["history"]
        ids = _zipf_ids(g, R, n, V)
        kw["history"] = (torch.arange(R + 1, dtype=torch.int32, device="cuda") * n, ids.reshape(-1).to(torch.int32))
        if case["rule"] == "chat":
            kw["repetition"] = f32(1.05)
        elif case["rule"] == "plain":
            kw.update(presence=f32(0.6), frequency=f32(0.2))
        else:
            kw.update(repetition=f32(1.1), presence=f32(0.5), frequency=f32(0.3))
    entries = case["bias"] + case.get("suppress", 0)
    if entries:
        # strictly increasing IDs: one per stratum of the vocabulary
        at = torch.arange(entries, device="cuda", dtype=torch.float64)[None, :] + _uniform(g, (R, entries))
        ids = (at * (V / entries)).long().clamp_(max=V - 1)
        ids = ids + torch.arange(entries, device="cuda")[None, :]
        ids = torch.minimum(ids, V - entries + torch.arange(entries, device="cuda")[None, :])
        vals = _uniform(g, (R, entries), -4.0, 4.0).float()
        vals[:, ::4] = -100.0
        if case.get("suppress"):
            vals[:, : case["suppress"]] = -math.inf
        kw["bias"] = (torch.arange(R + 1, dtype=torch.int32, device="cuda") * entries,
                      ids.reshape(-1).to(torch.int32), vals.reshape(-1).contiguous())
    if case["mask"]:
        kw["mask"] = _mask_words(g, R, V)
        kw["tokenizer_vocab"] = V
    return kw


def _pick_inputs(case, seed):
    g = _gen(seed)
    spread = 2.5 if case["logits"] == "text" or case["mask"] else 3.0 if case["rule"] == "topk" else 2.0
    x = _logits(g, case, spread)
    kw = _lists(g, case, _rules(g, case))
    if case["kind"] == "race":
        R = case["rows"]
        if case["whole"]:
            whole = torch.arange(R, device="cuda") % case["whole"] == 0
            for name, off in (("top_k", 0), ("top_p", 1.0), ("min_p", 0.0)):
                if name in kw:
                    kw[name] = torch.where(whole, torch.full_like(kw[name], off), kw[name])
        kw["race"] = (torch.randint(1 << 62, (R,), generator=g, device="cuda"),
                      torch.randint(4, (R,), generator=g, device="cuda").to(torch.int32),
                      torch.randint(30000, (R,), generator=g, device="cuda").to(torch.int32))
    return x, kw


def _topn_inputs(case, seed):
    return _logits(_gen(seed), dict(case, logits="normal"), 3.0)


def _spec_inputs(case, seed):
    """Target logits with 1 to 10 peaks per position; the draft model's are
    the target's with N(0, 0.5^2) noise, its tokens drawn from its softmax."""
    g = _gen(seed)
    R, K, V = case["rows"], case["draft"], case["vocab"]
    tgt = 2.0 * torch.randn((R, K + 1, V), generator=g, device="cuda")
    ids = torch.randint(V, (R, K + 1, 10), generator=g, device="cuda")
    amp = _uniform(g, (R, K + 1, 10), 4.0, 10.0).float()
    amp *= torch.arange(10, device="cuda") < torch.randint(1, 11, (R, K + 1, 1), generator=g, device="cuda")
    tgt.scatter_reduce_(2, ids, torch.gather(tgt, 2, ids) + amp, "amax")
    drf = tgt[:, :K] + 0.5 * torch.randn((R, K, V), generator=g, device="cuda")
    u = _uniform(g, (R, K, 1))
    cdf = torch.cumsum(torch.softmax(drf.double(), 2), 2)
    toks = torch.searchsorted(cdf, u * cdf[..., -1:]).clamp_(max=V - 1)[..., 0].to(torch.int32)
    return (tgt, drf, toks.contiguous(), _uniform(g, (R,), 0.7, 1.0), _uniform(g, (R, K)), _uniform(g, (R, K)),
            _uniform(g, (R,)))


def _lm_inputs(case, seed):
    """Normalised hidden states and a head whose logits spread like a
    model's (standard deviation about 2); a quarter of the rows greedy, the
    rest top_k 20, 50 and 100 with top_p and min_p."""
    g = _gen(seed)
    R, K, V = case["rows"], case["hidden"], case["vocab"]
    h = torch.randn((R, K), generator=g, device="cuda").to(torch.bfloat16)
    w = (torch.randn((V, K), generator=g, device="cuda") * (2.0 / math.sqrt(K))).to(torch.bfloat16)
    row = torch.arange(R, device="cuda")
    rule = dict(temperature=torch.where(row % 4 == 0, 0.0, _uniform(g, (R,), 0.3, 1.2)),
                top_k=torch.tensor([20, 20, 50, 100], dtype=torch.int32, device="cuda")[row % 4],
                top_p=_uniform(g, (R,), 0.7, 1.0), min_p=torch.full((R,), 0.02, dtype=torch.float64, device="cuda"),
                uniform=_uniform(g, (R,)))
    return h, w, rule


# ---------------------------------------------------------------------------
# What a program holds, and one pass

def prepare(case, seed):
    kind = case["kind"]
    st = dict(kind=kind)
    if kind == "topn":
        st["x"], st["n"], st["vocab"] = _topn_inputs(case, seed), case["n"], case["vocab"]
        st["s"] = Sampler(max_rows=case["rows"], max_vocab=case["vocab"])
    elif kind == "spec":
        tgt, drf, *rest = _spec_inputs(case, seed)
        st["s"] = Sampler(max_rows=case["rows"], max_vocab=case["vocab"])
        st["tgt"], st["drf"] = tgt, drf
        st["keep"], st["f"] = rest, st["s"].spec_launcher(tgt, drf, *rest)
    elif kind == "lm_head":
        h, w, rule = _lm_inputs(case, seed)
        st["s"] = s = Sampler(max_rows=case["rows"], max_vocab=case["vocab"])
        logits, tiles = s.lmhead(h, w, stats=True)
        st["keep"], st["logits"] = (h, w, rule, tiles), logits
        st["gemm"] = s.lmhead_launcher(h, w, logits, tiles)
        st["pick"] = s.finish_launcher(logits, tiles, **rule)
    else:
        x, kw = _pick_inputs(case, seed)
        st["s"] = s = Sampler(max_rows=case["rows"], max_vocab=case["vocab"])
        st["x"], st["keep"] = x, kw
        if kind == "step":
            st["f"] = s.step_launcher(x, n=case["n"], vocab=case["vocab"], **kw)
        else:
            st["f"] = s.launcher(x, vocab=case["vocab"], **kw)
    return st


def _picked(out):
    return dict(token=out.token, logprob=out.sampling_logprob, status=out.status, kept=out.kept_count)


def run(st):
    kind = st["kind"]
    if kind == "topn":
        ids, lps, mx, ln, status = st["s"].logsoftmax_topn(st["x"], st["n"], vocab=st["vocab"])
        return dict(ids=ids, logprobs=lps, maximum=mx, log_normalizer=ln, status=status)
    if kind == "spec":
        st["f"](st["tgt"], st["drf"])
        tokens, count, accepted, status = st["f"].out
        return dict(tokens=tokens, count=count, accepted=accepted, status=status)
    if kind == "lm_head":
        st["gemm"]()
        st["pick"]()
        return dict(logits=st["logits"], **_picked(st["pick"].out))
    st["f"](st["x"])
    out = _picked(st["f"].out)
    if kind == "step":
        r = st["f"].receipts
        out.update(ids=r.ids, logprobs=r.logprobs, token_logprob=r.token_logprob, receipt_status=r.status)
    return out


# ---------------------------------------------------------------------------
# What a pass cannot do without, and how near its results have to be

def work(case):
    R, V = case["rows"], case["vocab"]
    if case["kind"] == "spec":
        K = case["draft"]
        return dict(bytes=R * ((2 * K + 1) * V * 4 + K * (4 + 8 + 8) + 16 + (K + 1) * 4 + 12), flops=0)
    if case["kind"] == "lm_head":
        K = case["hidden"]
        return dict(bytes=2 * K * (V + R) + 4 * R * V + R * (28 + OUT_BYTES), flops=2 * R * K * V)
    n = R * V * (4 if case["dtype"] == "f32" else 2)
    if case["kind"] == "topn":
        return dict(bytes=n + R * (case["n"] * 12 + 20), flops=0)
    n += R * (4 * case["history"] + 8 * (case["bias"] + case.get("suppress", 0)) + 44 + OUT_BYTES)
    if case["mask"]:
        n += R * ((V + 31) // 32) * 4
    if case["kind"] == "step":
        n += R * (case["n"] * 12 + 12)
    if case["kind"] == "race":
        n += R * 16
    return dict(bytes=n, flops=0)


def tolerance(case):
    # Tokens, kept sets and statuses are certified decisions: none may differ.
    # A pick's log probability is f64 arithmetic over f64 sums (measured
    # against `exact`: 2e-16).  The log-softmax head and the receipts take
    # each weight from an f32 exp2 (measured 2e-10 and 4e-9 over the listed
    # batches, 2^-22 and 2^-20.9 for a single weight); the GEMM accumulates
    # its bf16 products in f32 (measured 2e-7, the log probabilities over its
    # logits 5e-7).
    return {"pick": {"rel": 1e-12}, "race": {"rel": 1e-12}, "topn": {"rel": 2e-7}, "step": {"rel": 2e-7},
            "spec": "exact", "lm_head": {"rel": 2e-6}}[case["kind"]]


# ---------------------------------------------------------------------------
# The same in plain torch, 64 bits

def _adjust(x, V, r, kw):
    """Row r's logits after bias and penalties: f32, each operation rounded."""
    l = x[r, :V].float().clone()
    sup = None
    if "bias" in kw:
        off, ids, vals = kw["bias"]
        b0, b1 = int(off[r]), int(off[r + 1])
        i, v = ids[b0:b1].long(), vals[b0:b1]
        sup = i[v == -math.inf]
        fin = v != -math.inf
        l[i[fin]] = l[i[fin]] + v[fin]
    if "history" in kw:
        off, ids = kw["history"]
        c = torch.bincount(ids[int(off[r]):int(off[r + 1])].long(), minlength=V)
        seen = torch.nonzero(c)[:, 0]
        at = lambda name, default: kw[name][r] if name in kw else torch.tensor(default, device=l.device)
        s = l[seen]
        s = torch.where(s < 0, s * at("repetition", 1.0), s / at("repetition", 1.0))
        s = s - c[seen].float() * at("frequency", 0.0)
        l[seen] = s - at("presence", 0.0)
    if sup is not None:
        l[sup] = torch.finfo(torch.float32).min
    return l


def _legal(kw, V, r, device):
    if "mask" not in kw:
        return torch.arange(V, device=device)
    w = kw["mask"][r].long() & 0xFFFFFFFF
    bits = (w[:, None] >> torch.arange(32, device=device)) & 1
    return torch.nonzero(bits.reshape(-1)[:V])[:, 0]


def _kept(l, T, top_k, top_p, min_p):
    """The kept flags of the compact legal row l (f64), and its weights."""
    n = l.numel()
    s = (l - l.max()) / T
    w = torch.exp(s)
    keep = torch.ones(n, dtype=torch.bool, device=l.device)
    k = top_k if 0 < top_k < n else 0
    if not (top_p >= 1.0 and k == 0):
        order = torch.sort(l, descending=True, stable=True).indices
        ws = w[order]
        if k:
            m, target = k, top_p * ws[:k].sum()
        else:
            total = w.sum()
            m, target = int((ws >= total * 1e-9).sum()), top_p * total
        cum = torch.cumsum(ws, 0)
        if not k and not bool(cum[m - 1] >= target):
            m = n
        hit = torch.nonzero(cum[:m] >= target)
        m = int(hit[0]) + 1 if hit.numel() else m
        keep = torch.zeros(n, dtype=torch.bool, device=l.device)
        keep[order[:m]] = True
    if min_p > 0.0:
        keep &= s >= math.log(min_p)
    return keep, s, w


def _race_bits(seed, choice, position, ids):
    """Philox4x32-10 words (hi, lo) of each token."""
    M = 0xFFFFFFFF
    c = [ids >> 1, torch.full_like(ids, position), torch.full_like(ids, choice), torch.full_like(ids, 0x72616365)]
    k0, k1 = seed & M, (seed >> 32) & M
    for i in range(10):
        if i:
            k0, k1 = (k0 + 0x9E3779B9) & M, (k1 + 0xBB67AE85) & M
        p0, p1 = 0xD2511F53 * c[0], 0xCD9E8D57 * c[2]
        c = [((p1 >> 32) & M) ^ c[1] ^ k0, p1 & M, ((p0 >> 32) & M) ^ c[3] ^ k1, p0 & M]
    odd = (ids & 1).bool()
    return torch.where(odd, c[2], c[0]), torch.where(odd, c[3], c[1])


def _gumbel(hi, lo):
    small = hi < 1 << 31
    bits = hi.double() * 4294967296.0 + lo.double()
    inv = (hi ^ 0xFFFFFFFF).double() * 4294967296.0 + (lo ^ 0xFFFFFFFF).double()
    scale = 2.0 ** -64
    e = torch.where(small, -torch.log1p(-((bits + 0.5) * scale)), -torch.log((inv + 0.5) * scale))
    return -torch.log(e)


def _exact_picks(x, V, kw):
    """token, logprob, status and kept count of every row, in 64 bits."""
    R, dev = x.shape[0], x.device
    out = dict(token=torch.zeros(R, dtype=torch.int32), logprob=torch.zeros(R, dtype=torch.float64),
               status=torch.zeros(R, dtype=torch.int32), kept=torch.zeros(R, dtype=torch.int32))
    at = lambda name, r, default: kw[name][r].item() if name in kw else default
    for r in range(R):
        l = _adjust(x, V, r, kw)
        ids = _legal(kw, V, r, dev)
        l = l[ids].double()
        T = at("temperature", r, 1.0)
        if T == 0.0:
            out["token"][r], out["kept"][r] = int(ids[torch.nonzero(l == l.max())[0, 0]]), 1
            continue
        keep, s, w = _kept(l, T, int(at("top_k", r, 0)), at("top_p", r, 1.0), at("min_p", r, 0.0))
        at_kept = torch.nonzero(keep)[:, 0]
        wk = w[at_kept]
        if "race" in kw:
            seed, choice, position = (int(t[r]) for t in kw["race"])
            score = l[at_kept] / T + _gumbel(*_race_bits(seed, choice, position, ids[at_kept]))
            j = int(torch.nonzero(score == score.max())[0, 0])
        else:
            cum = torch.cumsum(wk, 0)
            hit = torch.nonzero(at("uniform", r, 0.0) * wk.sum() < cum)
            j = int(hit[0, 0]) if hit.numel() else int(torch.nonzero(wk > 0)[-1, 0])
        out["token"][r] = int(ids[at_kept[j]])
        out["logprob"][r] = s[at_kept[j]] - torch.log(wk.sum())
        out["kept"][r] = at_kept.numel()
    return {k: v.to(dev) for k, v in out.items()}


def _exact_topn(l, n):
    """The log-softmax head of f32 rows l: ids, logprobs, maximum, ln(sum)."""
    ids = torch.sort(l, dim=1, descending=True, stable=True).indices[:, :n]
    d = l.double()
    mx = d.max(1).values
    ln = torch.log(torch.exp(d - mx[:, None]).sum(1))
    return ids.to(torch.int32), torch.gather(d, 1, ids) - mx[:, None] - ln[:, None], mx, ln


def _exact_spec(case, seed):
    tgt, drf, toks, T, ua, ur, ub = _spec_inputs(case, seed)
    R, K = case["rows"], case["draft"]
    dev = tgt.device
    out = torch.full((R, K + 1), -1, dtype=torch.int32)
    count, accepted = torch.zeros(R, dtype=torch.int32), torch.zeros(R, dtype=torch.int32)
    pick = lambda w, u: int(torch.nonzero(u * w.sum() < torch.cumsum(w, 0))[0, 0])
    for r in range(R):
        for j in range(K + 1):
            wt = torch.exp((tgt[r, j].double() - tgt[r, j].max().double()) / T[r])
            count[r] = j + 1
            if j == K:
                out[r, j] = pick(wt, ub[r])
                break
            wd = torch.exp((drf[r, j].double() - drf[r, j].max().double()) / T[r])
            p, q, t = wt / wt.sum(), wd / wd.sum(), int(toks[r, j])
            if bool(ua[r, j] < p[t] / q[t]):
                out[r, j], accepted[r] = t, j + 1
                continue
            out[r, j] = pick((p - q).clamp_(min=0.0), ur[r, j])
            break
    return dict(tokens=out.to(dev), count=count.to(dev), accepted=accepted.to(dev),
                status=torch.zeros(R, dtype=torch.int32, device=dev))


def exact(case, seed):
    kind, V = case["kind"], case["vocab"]
    if kind == "spec":
        return _exact_spec(case, seed)
    if kind == "topn":
        x = _topn_inputs(case, seed)
        parts = [_exact_topn(x[r:r + 16, :V].float(), case["n"]) for r in range(0, case["rows"], 16)]
        ids, lps, mx, ln = (torch.cat(p) for p in zip(*parts))
        return dict(ids=ids, logprobs=lps, maximum=mx, log_normalizer=ln,
                    status=torch.zeros(case["rows"], dtype=torch.int32, device=x.device))
    if kind == "lm_head":
        h, w, rule = _lm_inputs(case, seed)
        logits = torch.cat([h.double() @ w[v:v + 32768].double().t().contiguous() for v in range(0, V, 32768)], 1)
        # the f32 logits a correct GEMM rounds to decide the pick
        return dict(logits=logits, **_exact_picks(logits.float(), V, rule))
    x, kw = _pick_inputs(case, seed)
    out = _exact_picks(x, V, kw)
    if kind == "step":
        l = x[:, :V].float().clone()
        if "bias" in kw:
            off, ids, vals = kw["bias"]
            for r in range(case["rows"]):
                b = slice(int(off[r]), int(off[r + 1]))
                l[r, ids[b][vals[b] == -math.inf].long()] = torch.finfo(torch.float32).min
        ids, lps, mx, ln = _exact_topn(l, case["n"])
        tok = torch.gather(l.double(), 1, out["token"].long()[:, None])[:, 0]
        out.update(ids=ids, logprobs=lps, token_logprob=tok - mx - ln,
                   receipt_status=torch.zeros(case["rows"], dtype=torch.int32, device=x.device))
    return out
