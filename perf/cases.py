"""What the speed of this framework is measured on: the calls a serving engine
makes of it, through zllm_amd.engine, over the sizes that it serves.

Five kinds of case, by the entry point that a decode loop calls:

  sample  BatchSampler.run over packed rows: penalties, bias, bans, top-k,
          top-p, min-p, the draw, logprobs and uncertainty
  step    ByteDfa.mask over the rows' grammar states, then BatchSampler.run
          under the mask; with `drafts`, verify_drafts of the same rows on a
          second stream beside the sampler
  mask    ByteDfa.mask alone
  verify  verify_drafts alone: greedy (no draft logits) or rejection sampling
  lane    LaneBatcher.select: the batched lane's argmax, Gumbel or nucleus path

A context, a vocabulary's byte table and a compiled grammar are made once and
kept, as a server keeps them; logits, knobs, histories and grammar states come
from the seed. Sizes are those of bench.py's configurations and of the tests,
or generic ones between them (V from 20,000 to 151,936, 1 to 256 rows).
"""
import functools

import numpy as np
import torch

from zllm_amd import grammar as G
from zllm_amd import synth
from zllm_amd.engine import (BatchSampler, ByteDfa, Context, DecodeControl, LaneBatcher, LaneSeq, LogitFSM,
                             PenaltyConfig, RowRequest, SamplerConfig, SamplingParams, TokenByteTable, verify_drafts)

TOP_STRIDE = 20   # the width of the top_logprobs outputs (the OpenAI cap, BatchSampler.run's default)


def listed():
    return [
        # one chat request alone: the smallest call, where launches and latency are all there is
        dict(name="chat_one", kind="sample", rows=1, vocab=32000, knobs="chat"),
        # a greedy batch of the batched lane on an odd vocabulary: one short launch
        dict(name="lane_greedy_few", kind="lane", rows=8, vocab=50257, path="argmax"),
        # an ordinary server batch of unconstrained requests with knobs of their own
        dict(name="batch_mixed", kind="sample", rows=64, vocab=128256, knobs="mixed"),
        # every option the API has, row by row, on an odd batch over an odd vocabulary
        dict(name="options_ragged", kind="sample", rows=23, vocab=100003, knobs="all"),
        # regex-constrained plain sampling (T = 1, no cuts); the rows are in
        # states that were met before, as inside a long match
        dict(name="regex_step", kind="step", rows=32, vocab=128256, knobs="open", grammar="random", states=64,
             fresh=False, share=1.0, drafts=0),
        # schema-constrained output with a ban list; every state met for the first time
        dict(name="json_step", kind="step", rows=128, vocab=151936, knobs="nucleus_bans", grammar="json",
             states=2048, fresh=True, share=1.0, drafts=0),
        # the full continuous-batching step: half the rows under a grammar,
        # speculative verification beside the sampler
        dict(name="full_step", kind="step", rows=256, vocab=151936, knobs="mixed", grammar="json", states=512,
             fresh=True, share=0.5, drafts=4),
        # the mask of the response_format "any JSON" grammar, its states met for the first time
        dict(name="mask_any_json", kind="mask", rows=128, vocab=151936, grammar="any_json", states=0, fresh=True),
        # greedy verification of n-gram drafts for a few requests
        dict(name="verify_greedy_few", kind="verify", rows=4, vocab=32000, drafts=8, sampled=False),
        # rejection sampling against a draft model
        dict(name="verify_sampled", kind="verify", rows=64, vocab=128256, drafts=4, sampled=True),
        # the batched lane with top-k / top-p knobs: top-64 pool and nucleus draw
        dict(name="lane_nucleus", kind="lane", rows=256, vocab=151936, path="topk"),
        # the batched lane with temperatures only, an ordinary batch
        dict(name="lane_gumbel", kind="lane", rows=96, vocab=128256, path="sample"),
    ]


def draw(rng):
    kind = rng.choice(["sample", "sample", "step", "step", "mask", "verify", "lane"])
    rows = max(1, min(256, round(2.0 ** rng.uniform(0.0, 8.0))))
    vocab = rng.randrange(20000, 151937)
    case = dict(kind=kind, rows=rows, vocab=vocab)
    if kind == "sample":
        case.update(knobs=rng.choice(["chat", "mixed", "open", "nucleus_bans", "all"]))
    elif kind in ("step", "mask"):
        g = rng.choice(["random", "json", "any_json"])
        case.update(grammar=g, states={"random": rng.randrange(16, 257), "json": rng.randrange(128, 2049),
                                       "any_json": 0}[g], fresh=rng.random() < 0.5)
        if kind == "step":
            case.update(knobs=rng.choice(["chat", "mixed", "open", "nucleus_bans", "all"]),
                        share=rng.choice([0.25, 0.5, 1.0]), drafts=rng.choice([0, 0, 2, 4]))
            if case["drafts"]:
                case["rows"] = min(rows, 192)   # no more work than the full step's
    elif kind == "verify":
        # the logits of up to 2 * drafts + 1 positions a row: no more of them than the full step has
        case.update(drafts=rng.randrange(1, 9), sampled=rng.random() < 0.6)
        case["rows"] = max(1, min(rows, 256 * 9 // (2 * case["drafts"] + 1)))
    else:
        case.update(path=rng.choice(["argmax", "sample", "topk"]))
    return case


# ---------------------------------------------------------------- inputs
@functools.lru_cache(maxsize=None)
def _context(rows, vocab):
    return Context(0, rows, vocab)


@functools.lru_cache(maxsize=None)
def _vocabulary(V):
    """Token byte strings as synth.synthetic_vocab describes them (lengths 1
    to 16, geometric with mean 4; 70% ASCII, 20% space-prefixed words, 10%
    UTF-8 continuation bytes), all bytes drawn at once: (offsets, bytes)."""
    rng = np.random.default_rng(V)
    lens = np.minimum(rng.geometric(0.25, size=V), 16)
    offs = np.zeros(V + 1, np.uint32)
    offs[1:] = np.cumsum(lens)
    n = int(offs[-1])
    kind = np.repeat(rng.random(V), lens)
    word = rng.integers(97, 123, n)
    word[offs[:-1].astype(np.int64)] = 32
    data = np.where(kind < 0.7, rng.integers(33, 127, n), np.where(kind < 0.9, word, rng.integers(0x80, 0xC0, n)))
    return offs, data.astype(np.uint8)


@functools.lru_cache(maxsize=None)
def _table(rows, V):
    offs, data = _vocabulary(V)
    return TokenByteTable.from_csr(_context(rows, V), offs, data, np.ones(V, np.uint8), eos=V - 1)


@functools.lru_cache(maxsize=None)
def _any_json():
    g = G.HostDfa(G.any_json_regex_default())
    return np.asarray(g.trans).reshape(-1, 256), np.asarray(g.dead), np.asarray(g.accept)


def _automaton(case, seed):
    """(trans [S, 256], dead [S], accept [S]) of the case's grammar."""
    if case["grammar"] == "random":
        return synth.random_dfa(case["states"], seed, dead_rate=0.3)
    if case["grammar"] == "json":
        return synth.json_dfa(case["states"], seed)
    return _any_json()


def _live(trans, dead, accept):
    """States from which an accepting state can be reached."""
    live = (accept != 0) & (dead == 0)
    while True:
        more = (live | live[trans].any(axis=1)) & (dead == 0)
        if (more == live).all():
            return live
        live = more


def _row_states(case, seed, trans, dead, accept):
    """Current grammar state per row, -1 on the rows without a grammar."""
    rng = np.random.default_rng(seed + 17)
    B = case["rows"]
    st = rng.choice(np.nonzero(_live(trans, dead, accept))[0], B).astype(np.int32)
    free = np.arange(B) * case.get("share", 1.0) % 1.0 >= case.get("share", 1.0)
    st[free] = -1
    return st


def _generator(seed):
    return torch.Generator(device="cuda").manual_seed(seed)


def _logits(B, V, seed, spikes=16):
    """N(0, 2) with a power-law peak of `spikes` ids (synth.logits_powerlaw's
    distribution), rows padded to a multiple of 4 as the ABI asks."""
    g = _generator(seed)
    x = torch.zeros((B, (V + 3) // 4 * 4), device="cuda")[:, :V]
    x.copy_(torch.randn((B, V), device="cuda", generator=g) * 2.0)
    ids = torch.randint(0, V, (B, spikes), device="cuda", generator=g)
    peak = 15.0 * torch.arange(1, spikes + 1, device="cuda").float() ** -1.2
    x.scatter_add_(1, ids, peak.expand(B, spikes))
    return x


def _history(rng, V, n):
    """A count map over the last n tokens; a few of them keep coming back."""
    h = np.concatenate([rng.integers(0, V, n - n // 4), rng.choice(rng.integers(0, V, 8), n // 4)])
    ids, cnt = np.unique(h, return_counts=True)
    return dict(zip(ids.tolist(), cnt.tolist()))


def _rows(case, seed, masked):
    """One RowRequest per row with the case's knobs."""
    rng = np.random.default_rng(seed + 29)
    V, out = case["vocab"], []
    for i in range(case["rows"]):
        knobs = case["knobs"]
        rest = dict(logprobs=True, detect_hallucination=True, top_logprobs=5)
        pen, bias, fsm, hist = PenaltyConfig(), (), None, 0
        if knobs == "all":
            knobs = ["chat", "mixed", "open", "min_p", "greedy", "bias", "nucleus_bans", "wide_k"][(i + seed) % 8]
            wants = int(rng.integers(0, 4))   # observers: none, logprobs, uncertainty, both
            rest = dict(logprobs=bool(wants & 1), detect_hallucination=bool(wants & 2),
                        top_logprobs=int(rng.choice([0, 1, 5, 20])) if wants & 1 else 0)
        if knobs == "chat":
            cfg, pen, hist = SamplerConfig(0.8, 40, 0.95, 0.0), PenaltyConfig(repeat=1.1), 64
        elif knobs == "mixed":
            cfg = SamplerConfig(float(rng.uniform(0.5, 1.2)), int(rng.choice([0, 20, 50])),
                                float(rng.uniform(0.8, 1.0)), 0.0)
            pen, hist = PenaltyConfig(1.0, float(rng.uniform(0, 0.5)), float(rng.uniform(0, 0.5))), 256
        elif knobs == "open":
            cfg = SamplerConfig(1.0, 0, 1.0, 0.0)
        elif knobs == "min_p":
            cfg = SamplerConfig(float(rng.uniform(0.7, 1.5)), 0, 1.0, float(rng.uniform(0.02, 0.1)))
        elif knobs == "greedy":
            cfg, pen, hist = SamplerConfig(0.0, 0, 1.0, 0.0), PenaltyConfig(repeat=1.05), 512
        elif knobs == "bias":
            cfg = SamplerConfig(0.9, 0, 0.9, 0.0)
            bias = [(int(t), float(b)) for t, b in zip(rng.integers(0, V, 60), rng.uniform(-8, 4, 60))]
        elif knobs == "nucleus_bans":
            cfg = SamplerConfig(0.7, 0, 0.9, 0.0)
            fsm = LogitFSM(banned=rng.choice(V, 500, replace=False))
        else:   # wide_k: more survivors than any candidate list holds
            cfg = SamplerConfig(1.1, int(rng.integers(200, 2000)), 0.98, 0.01)
        ctrl = DecodeControl(pen, bias, seed=int(rng.integers(0, 2**62)))
        ctrl.counter = int(rng.integers(0, 4096))
        if hist:
            ctrl.counts = _history(rng, V, hist)
        out.append(RowRequest(cfg, ctrl, fsm, masked=bool(masked[i]), **rest))
    return out


def _drafts(case, seed, sampled):
    """Target logits [B, k+1, V] with a peak per position and draft ids that
    are mostly that peak; draft logits are the target's with noise."""
    B, V, k = case["rows"], case["vocab"], case["drafts"]
    g = _generator(seed + 99)
    ld = (V + 3) // 4 * 4
    peak = torch.randint(0, V, (B, k + 1, 1), device="cuda", generator=g)
    target = torch.zeros((B, k + 1, ld), device="cuda")[:, :, :V]
    target.copy_(torch.randn((B, k + 1, V), device="cuda", generator=g) * 2.0)
    target.scatter_add_(2, peak, torch.full((B, k + 1, 1), 12.0, device="cuda"))
    ids = peak[:, :k, 0].to(torch.int32)
    draft = None
    if sampled:
        draft = torch.zeros((B, k, ld), device="cuda")[:, :, :V]
        draft.copy_(target[:, :k] + torch.randn((B, k, V), device="cuda", generator=g) * 0.5)
    else:
        # an n-gram draft is wrong now and then
        miss = torch.rand((B, k), device="cuda", generator=g) < 0.2
        ids = torch.where(miss, torch.randint(0, V, (B, k), device="cuda", generator=g).to(torch.int32), ids)
    T = torch.rand(B, device="cuda", generator=g) * 0.7 + 0.5 if sampled else torch.zeros(B, device="cuda")
    return dict(target=target, draft=draft, ids=ids.contiguous(), T=T,
                seed=torch.arange(B, dtype=torch.int64, device="cuda") + 5000 + seed,
                counter=torch.zeros(B, dtype=torch.int64, device="cuda"))


@functools.lru_cache(maxsize=None)
def _second_stream():
    return torch.cuda.Stream()


def prepare(case, seed):
    B, V, kind = case["rows"], case["vocab"], case["kind"]
    S = dict(case=case, ctx=_context(B, V))
    if kind in ("sample", "step", "lane"):
        S["logits"] = _logits(B, V, seed)
    if kind in ("step", "mask"):
        trans, dead, accept = _automaton(case, seed)
        st = _row_states(case, seed, trans, dead, accept)
        S.update(table=_table(B, V), dfa=ByteDfa(S["ctx"], trans, dead, accept), states=torch.from_numpy(st).cuda(),
                 bits=torch.empty((B, (V + 31) // 32), dtype=torch.int32, device="cuda"))
        masked = st >= 0
    else:
        masked = np.zeros(B, bool)
    if kind in ("sample", "step"):
        S["sampler"] = BatchSampler(S["ctx"])
        S["bufs"] = S["sampler"].pack(S["logits"], _rows(case, seed, masked))
    if kind == "verify" or case.get("drafts"):
        S["drafts"] = _drafts(case, seed, case.get("sampled", True))
    if kind == "step" and case["drafts"]:
        S["event"] = torch.cuda.Event()
        S["event"].record()
    if kind == "lane":
        rng = np.random.default_rng(seed + 41)
        S["lane"] = LaneBatcher(S["ctx"])
        for i in range(B):
            temp = 0.0 if case["path"] == "argmax" else float(rng.uniform(0.5, 1.2))
            top_k, top_p = 0, 1.0
            if case["path"] == "topk":
                top_k, top_p = int(rng.choice([0, 20, 50])), float(rng.uniform(0.8, 1.0))
            seq = LaneSeq(i, SamplingParams(temp, top_k, top_p), int(rng.integers(0, 2**32)), V - 1, 1 << 20)
            seq.generated = [0] * int(rng.integers(1, 64))
            S["lane"].add(seq)
    return S


# ---------------------------------------------------------------- one pass
def _mask(S):
    if S["case"]["fresh"]:
        S["dfa"].memo_clear()   # the first step of these states: no bitset of an earlier one serves
    return S["dfa"].mask(S["table"], S["states"], S["case"]["vocab"], out=S["bits"])


def _verify(S):
    d = S["drafts"]
    return verify_drafts(S["ctx"], d["target"], d["ids"], d["T"], d["seed"], d["counter"], d["draft"])


def run(S):
    kind = S["case"]["kind"]
    if kind == "sample":
        return S["sampler"].run(S["logits"], S["bufs"], top_stride=TOP_STRIDE)
    if kind == "mask":
        return _mask(S)
    if kind == "verify":
        return _verify(S)
    if kind == "lane":
        return S["lane"].select(S["logits"])
    if not S["case"]["drafts"]:
        bits = _mask(S)
        return dict(bits=bits, **S["sampler"].run(S["logits"], S["bufs"], bits, top_stride=TOP_STRIDE))
    # the verification is independent of this step's sampling: on a second
    # stream from where the sampler's kernels begin
    main, other = torch.cuda.current_stream(), _second_stream()
    other.wait_stream(main)
    bits = _mask(S)
    out = S["sampler"].run(S["logits"], S["bufs"], bits, top_stride=TOP_STRIDE, pass_event=S["event"])
    with torch.cuda.stream(other):
        other.wait_event(S["event"])
        accepted, nxt = _verify(S)
    main.wait_stream(other)
    for t in (accepted, nxt):
        t.record_stream(main)
    return dict(bits=bits, accepted=accepted, next=nxt, **out)


# ---------------------------------------------------------------- what it has to be
def work(case):
    """Each logit read once, each list and each output once. Operations: per
    logit of the sampler a comparison, an exponential, two sums and a product
    (10 counted); of the Gumbel lane a hash and two logarithms (20); of a
    stochastic verification an exponential and a sum (4); else a comparison."""
    B, V, kind = case["rows"], case["vocab"], case["kind"]
    nbytes = flops = 0
    words = (V + 31) // 32 * 4
    if kind in ("sample", "step"):
        lists = {"chat": 64 * 8, "mixed": 256 * 8, "open": 0, "nucleus_bans": 2000, "all": 1000}[case["knobs"]]
        nbytes += B * (4 * V + lists + 40 + 16 + 7 * 4 + 8 * 5)
        flops += B * V * 10
    if kind in ("step", "mask"):
        rows = round(B * case.get("share", 1.0))
        offs, data = _vocabulary(V)
        nbytes += B * (4 + words) + (len(data) + V)
        if kind == "step":
            nbytes += rows * words
        flops += rows * V
    drafts = case.get("drafts", 0)
    if drafts:
        sampled = case.get("sampled", True)
        n = (2 if sampled else 1) * drafts + 1
        nbytes += B * (n * 4 * V + 4 * drafts + 28)
        flops += B * n * V * (4 if sampled else 1)
    if kind == "lane":
        nbytes += B * (4 * V + 24)
        flops += B * V * (20 if case["path"] == "sample" else 1)
    return dict(bytes=nbytes, flops=flops)


def tolerance(case):
    """Ids, counts and bitsets are fixed by the reference's operation order,
    which this path reproduces: they are equal. The floats are logarithms,
    quotients and differences of those exact f32 sums: one unit in the last
    place of a logarithm apart at most (6e-8), relative to values near 1."""
    if case["kind"] in ("sample", "step"):
        return {"rel": 1e-6, "max": 1e-5, "differ": 0.0}
    return "exact"


def _allowed(case, seed, states, trans, dead, accept):
    """bool [B, V]: the ids the grammar allows per row, by a plain walk."""
    V = case["vocab"]
    offs, data = _vocabulary(V)
    live = torch.from_numpy(_live(trans, dead, accept)).cuda()
    alive = torch.from_numpy(dead == 0).cuda()
    t = torch.from_numpy(trans.astype(np.int64)).cuda().reshape(-1)
    start = torch.from_numpy(offs[:-1].astype(np.int64)).cuda()
    lens = torch.from_numpy(np.diff(offs).astype(np.int64)).cuda()
    byts = torch.from_numpy(np.concatenate([data, np.zeros(16, np.uint8)]).astype(np.int64)).cuda()
    out = torch.ones((len(states), V), dtype=torch.bool, device="cuda")
    for r, s in enumerate(states.tolist()):
        if s < 0:
            continue
        cur = torch.full((V,), s, dtype=torch.int64, device="cuda")
        ok = torch.ones(V, dtype=torch.bool, device="cuda")
        for j in range(int(lens.max())):
            on = lens > j
            cur = torch.where(on & ok, t[cur * 256 + byts[start + j]], cur)
            ok &= alive[cur]
        ok &= live[cur]
        ok[V - 1] = False
        ok[V - 1] = bool(accept[s]) or not bool(ok.any())
        out[r] = ok
    return out


def exact(case, seed):
    """The observers' numbers in 64 bits (the sampler's token and what hangs
    on it are whole numbers of an f32 operation order: no such value)."""
    if case["kind"] not in ("sample", "step"):
        return None
    B, V = case["rows"], case["vocab"]
    allow = None
    masked = np.zeros(B, bool)
    if case["kind"] == "step":
        auto = _automaton(case, seed)
        st = _row_states(case, seed, *auto)
        allow, masked = _allowed(case, seed, st, *auto), st >= 0
    x = _logits(B, V, seed)
    rows = _rows(case, seed, masked)
    top_lps = torch.zeros((B, TOP_STRIDE), dtype=torch.float64, device="cuda")
    entropy, max_prob, margin = (torch.full((B,), float("nan"), dtype=torch.float64, device="cuda") for _ in range(3))
    for i, rq in enumerate(rows):
        y = x[i].double()
        if rq.fsm is not None:
            y[torch.tensor(rq.fsm.banned, device="cuda")] = -float("inf")
        if allow is not None:
            y[~allow[i]] = -float("inf")
        lp = y - y.max() - (y - y.max()).exp().sum().log()
        p = lp.exp()
        if rq.top_logprobs:
            top_lps[i, :rq.top_logprobs] = lp.topk(rq.top_logprobs).values
        if rq.detect_hallucination:
            two = p.topk(2).values
            entropy[i] = -(p * torch.where(p > 0, lp, torch.zeros_like(lp))).sum()
            max_prob[i], margin[i] = two[0], two[0] - two[1]
    out = dict(token=None, logprob=None, top_ids=None, top_lps=top_lps, top_n=None, entropy=entropy,
               max_prob=max_prob, margin=margin, chosen_lp=None, status=None)
    if allow is not None:
        out["bits"] = None
        if case["drafts"]:
            out.update(accepted=None, next=None)
    return out
