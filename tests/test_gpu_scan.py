"""The row kernel's lists from group maxima (zs_k_scan): rows where the groups
of 16, 32 or 64 ids, their thresholds or the listed groups can go wrong, at
the widths where the group size changes, compared with the oracle (tokens and
top ids bit for bit, floats within gpu_util.compare's 1e-5)."""
import numpy as np
import pytest

from tests.gpu_util import compare, oracle_row, run_gpu

pytestmark = pytest.mark.gpu


def _case(V):
    rng = np.random.default_rng(V)
    B = 20
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    P = [dict(temperature=0.9, top_k=40, top_p=0.95, top_logprobs=20, seed=i) for i in range(B)]
    x[0].sort()                                    # the top entries adjacent: whole groups pass the threshold
    x[1] = 1.5                                     # every group at the threshold
    x[2, -3:] = [9.0, 11.0, 10.0]                  # the last, partial group
    x[3, V // 2:V // 2 + 200] = 20.0               # more equal entries than k, adjacent
    x[4] = -np.inf                                 # fewer ids above -inf than candidates
    x[4, [0, 70, V - 1]] = [1.0, 2.0, 0.5]
    x[5] = -np.inf                                 # 600 survivors, most in a few groups
    x[5, 100:700] = rng.normal(0, 1, 600)
    P[5].update(top_k=0)
    x[6] = -np.inf                                 # 500 survivors spread over the row
    x[6, rng.choice(V, 500, replace=False)] = rng.normal(0, 3, 500).astype(np.float32)
    P[6].update(top_k=0, min_p=0.01)
    for i, k in ((7, 129), (8, 300), (9, 511), (10, 512), (11, 1500), (12, V - 5)):
        P[i].update(top_k=k, top_p=0.97)           # larger k: by sorted list, by keys alone, by the big-row engine
    top = np.argsort(-x[13])[:64]                  # bans and biases in the top groups
    P[13].update(ban=[int(t) for t in top[:30]], bias=[(int(top[40]), 9.0), (int(top[41]), -9.0), (7, 30.0), (7, -4.0)])
    P[14].update(counts=[(int(t), int(c)) for t, c in zip(rng.choice(V, 1500, replace=False), rng.integers(1, 4, 1500))],
                 presence=0.4, frequency=0.3, repeat=1.2)   # lists longer than the registers hold
    x[15, [5, V // 3, V - 2]] = 30.0               # greedy: the last of the equal maxima
    P[15].update(temperature=0.0)
    x[16] = np.where(rng.random(V) < 0.5, np.float32(0.0), np.float32(-0.0))   # zeros of both signs at the threshold
    x[17, 11] = np.nan                             # a NaN
    x[18, V // 2] = np.inf
    P[19].update(temperature=0.0, counts=[(int(np.argmax(x[19])), 1)], presence=50.0)   # greedy, the maximum penalised
    return x, P


@pytest.mark.parametrize("V", [4095, 4096, 4099, 50257, 81920, 81921, 151936, 163844])
def test_lists_from_group_maxima(V):
    x, params = _case(V)
    print(f"[case] group maxima V={V}", flush=True)
    errs = compare(x, params, _run_padded(x, params))
    assert not errs, "\n".join(errs[:20])


def _run_padded(x, params, allow=None):
    """run_gpu for widths that are no multiple of 4 (rows padded in memory)."""
    import torch

    from tests.gpu_util import ctx, make_rows
    from zllm_amd.engine import BatchSampler
    B, V = x.shape
    c = ctx(max(64, B), max(151936, V))
    xs = torch.zeros((B, (V + 3) // 4 * 4), device="cuda")
    xs[:, :V] = torch.from_numpy(x)
    bs = BatchSampler(c)
    ab = torch.from_numpy(allow).cuda() if allow is not None else None
    out = bs.run(xs[:, :V], bs.pack(xs[:, :V], make_rows(params)), ab)
    torch.cuda.synchronize()
    return {k: v.cpu().numpy() for k, v in out.items()}


@pytest.mark.parametrize("V", [4096, 50257, 151936])
def test_lists_under_masks(V):
    """Allowed sets of 0 to most of the row, adjacent (all in the groups of a
    few waves) and spread, gathered and not, with bans and penalties inside."""
    rng = np.random.default_rng(V + 1)
    sizes = [1, 20, 27, 28, 300, 512, 513, 1000, 1024, 2048, 2049, min(V // 2, 30000)]
    B = 2 * len(sizes)
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    allow = np.zeros((B, V), bool)
    P = []
    for i in range(B):
        n = sizes[i // 2]
        ids = rng.choice(V, n, replace=False) if i % 2 else (np.arange(n) + V // 3) % V
        allow[i, ids] = True
        P.append(dict(temperature=[0.8, 1.0, 0.0][i % 3], top_k=[0, 30, 400][i // 3 % 3], top_p=0.9, top_logprobs=20,
                      seed=i, masked=True, ban=[int(t) for t in ids[:n // 10]],
                      counts=[(int(t), 1) for t in ids[n // 2:n // 2 + 40]], presence=0.5))
    bits = np.zeros((B, (V + 31) // 32), np.uint32)
    for i in range(B):
        b = np.packbits(np.pad(allow[i], (0, -V % 32)), bitorder="little")
        bits[i] = b.view(np.uint32)
    print(f"[case] group maxima under masks V={V}", flush=True)
    out = _run_padded(x, P, bits.view(np.int32))
    refs = [oracle_row(x[i], P[i], allow[i]) for i in range(B)]
    errs = compare(x, P, out, allow=allow, refs=refs)
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("V", [4092, 151936])
def test_zeros_of_both_signs(V):
    """A row of zeros of both signs: the first threshold is the key of +0,
    which the value below it must not turn away."""
    rng = np.random.default_rng(V)
    x = np.where(rng.random((4, V)) < 0.5, np.float32(0.0), np.float32(-0.0))
    params = [dict(temperature=0.9, top_k=k, top_p=0.95, top_logprobs=20, seed=i) for i, k in enumerate((40, 128, 0, 3))]
    print(f"[case] zeros of both signs V={V}", flush=True)
    errs = compare(x, params, run_gpu(x, params))
    assert not errs, "\n".join(errs)


@pytest.mark.parametrize("top_p", [1.0, 0.9])
def test_min_p_kept_lists(top_p):
    """The kept mass of min-p rows from per-wave lists (zs_k_big): 1 kept
    value, a stretch of the row (1280 ids) that keeps exactly as many as its
    list holds (512) and one more, kept values over all stretches, and a row
    that keeps everything; min_p above 1 keeps nothing."""
    V = 20000
    rng = np.random.default_rng(5)
    x = rng.normal(-12, 1, (7, V)).astype(np.float32)
    x[0, 17] = 9.0
    for i, n in ((1, 512), (2, 513)):
        x[i, 1280 + rng.choice(1280, n, replace=False)] = rng.normal(8, 0.3, n).astype(np.float32)
    x[3, rng.choice(V, 700, replace=False)] = rng.normal(8, 0.5, 700).astype(np.float32)
    x[4] = rng.normal(0, 0.1, V).astype(np.float32)
    x[5, :700] = 3.0
    params = [dict(temperature=1.1, top_k=0, top_p=top_p, min_p=0.05, seed=i, top_logprobs=3) for i in range(7)]
    params[6]["min_p"] = 1.5
    print(f"[case] min-p kept lists top_p={top_p}", flush=True)
    errs = compare(x, params, run_gpu(x, params))
    assert not errs, "\n".join(errs)


# per width: three quarters of the groups and one more, and the largest k whose
# ids are expected to fit the list and one more
@pytest.mark.parametrize("V,ks", [(4096, (129, 192, 193, 511)), (20000, (511, 512, 937, 938, 1200)), (32000, (1500, 1501)),
                                  (100003, (2304, 2305, 2400)), (128256, (2500, 2594, 2595, 3073))])
def test_wide_top_k(V, ks):
    rng = np.random.default_rng(V)
    x = rng.normal(0, 2, (2 * len(ks), V)).astype(np.float32)
    params = [dict(temperature=1.1, top_k=k, top_p=0.98, min_p=0.01 * (i % 2), top_logprobs=20, seed=i)
              for i, k in enumerate(np.repeat(ks, 2).tolist())]
    print(f"[case] wide top-k V={V}", flush=True)
    errs = compare(x, params, _run_padded(x, params))
    assert not errs, "\n".join(errs[:20])


def test_wide_top_k_lists_that_overflow():
    """More values at the threshold than the sampler's list holds, with the
    observers' candidates above them (rows 0 to 4) or among them: k up to 128
    takes the ones above and the k-th, larger k keep the observers' list alone;
    without observers nothing else is listed."""
    V = 50257
    rng = np.random.default_rng(8)
    P = [dict(temperature=1.0, top_k=k, top_p=0.9, top_logprobs=20, seed=i)
         for i, k in enumerate((100, 300, 511, 700, 300, 60, 61, 20, 128))]
    P[4].update(logprobs=False, detect_hallucination=False, top_logprobs=0)
    x = rng.normal(0, 1, (len(P), V)).astype(np.float32)
    for i in range(len(P)):
        x[i, 16 * 1000:16 * 1400] = 9.0                       # 400 groups of 16 equal values
        n = 60 if i < 7 else 5
        x[i, rng.choice(16000, n, replace=False)] = rng.uniform(10, 12, n).astype(np.float32)
    print("[case] wide top-k overflow", flush=True)
    errs = compare(x, P, _run_padded(x, P))
    assert not errs, "\n".join(errs)


@pytest.mark.parametrize("V", [20001, 50257, 128256, 163844])
def test_many_groups_at_a_threshold(V):
    """Rows of few distinct values, where most groups reach a threshold: the
    observers' ties by id, the sampler's k-th value at, above and below the
    tied value, k of every kind of list, ties under masks, bans and counts."""
    rng = np.random.default_rng(V)
    B = 22
    x = np.full((B, V), 1.5, np.float32)
    P = [dict(temperature=0.9, top_k=40, top_p=0.95, top_logprobs=20, seed=i) for i in range(B)]
    allow = np.ones((B, V), bool)
    for i, k in ((1, 1), (2, 128), (3, 300), (4, 511), (5, 600), (6, 900), (7, 0)):
        P[i].update(top_k=k)
    for i, n in ((8, 10), (9, 39), (10, 40), (11, 41), (12, 200)):
        x[i, rng.choice(V, n, replace=False)] = rng.uniform(2, 5, n).astype(np.float32)   # above the tied value
    x[13] = rng.integers(0, 3, V).astype(np.float32)                  # three values, the largest in most groups
    x[14] = np.where(rng.random(V) < 0.5, 0.0, -0.0).astype(np.float32)
    x[14, ::16] = 1.0                                                 # one id per group of 16
    x[15, :V // 2] = -np.inf                                          # ties in the second half alone
    P[16].update(ban=rng.choice(V, 700, replace=False).tolist(), counts=[(int(t), 2) for t in rng.choice(V, 900, replace=False)],
                 presence=0.5)
    P[17].update(temperature=0.0)                                     # greedy: the last id
    P[18].update(masked=True)
    allow[18] = rng.random(V) < 0.5
    P[19].update(masked=True, top_k=600)
    allow[19] = rng.random(V) < 0.9
    allow[19, :V // 3] = False
    x[20] = -np.finfo(np.float32).max                                 # the value next to -inf
    P[21].update(logprobs=False, detect_hallucination=False, top_logprobs=0)
    bits = np.zeros((B, (V + 31) // 32), np.uint32)
    for i in range(B):
        bits[i] = np.packbits(np.pad(allow[i], (0, -V % 32)), bitorder="little").view(np.uint32)
    print(f"[case] ties V={V}", flush=True)
    refs = [oracle_row(x[i], P[i], allow[i] if P[i].get("masked") else None) for i in range(B)]
    errs = compare(x, P, _run_padded(x, P, bits.view(np.int32)), refs=refs)
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("V", [4096, 50257, 128256, 163841])
def test_nan_in_a_group(V):
    """The greedy fold after the last NaN, which lies first, last, in the middle
    and next to others in its group, in the last group, at a penalised or
    biased id, under a mask or a ban (no NaN then), before values at -inf, ties
    and larger values in front of it; sampled rows beside them."""
    rng = np.random.default_rng(V)
    gs = 16 if V <= 81920 else 32 if V <= 163840 else 64
    g0 = V // 2 // gs * gs                                            # a group's first id
    at = [[g0], [g0 + gs - 1], [g0 + 5], [g0, g0 + 3, g0 + 9], [V - 1], [V - 2], [0], list(range(g0, g0 + gs)),
          [3, g0 + 2], [g0 + 4], [g0 + 4], [g0 + 4], [g0 + 4], [g0 + 4], [g0 + 4], [g0 + 4, V - 9]]
    B = 2 * len(at)
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    P = [dict(temperature=0.0 if i < len(at) else 0.9, top_k=[40, 0, 700][i % 3], top_p=0.95, top_logprobs=5, seed=i) for i in range(B)]
    allow = np.ones((B, V), bool)
    for i in range(B):
        k = i % len(at)
        x[i, at[k]] = np.nan
        if k == 9:
            x[i, g0 + 5:] = -np.inf                                   # nothing above -inf follows
        elif k == 10:
            x[i, g0 + 5:] = np.where(rng.random(V - g0 - 5) < 0.5, 0.0, -0.0)   # ties of both zeros follow
        elif k == 11:
            P[i].update(counts=[(g0 + 4, 2), (g0 + 6, 1), (V - 1, 1)], presence=0.5, bias=[(g0 + 7, 20.0), (g0 + 4, 1.0)])
        elif k == 12:
            P[i].update(ban=[g0 + 4, g0 + 5])                         # a banned NaN is none
        elif k == 13:
            P[i].update(masked=True)
            allow[i] = rng.random(V) < 0.5
            allow[i, g0 + 4] = i >= len(at)                           # masked out, and not
        elif k == 14:
            x[i, g0 + 4] = np.inf                                     # inf - inf: NaN in y alone
            P[i].update(bias=[(g0 + 4, -np.inf)])
        elif k == 15:
            x[i, :V - 9] += 40.0                                      # larger values in front of it
    bits = np.zeros((B, (V + 31) // 32), np.uint32)
    for i in range(B):
        bits[i] = np.packbits(np.pad(allow[i], (0, -V % 32)), bitorder="little").view(np.uint32)
    print(f"[case] NaN in a group V={V}", flush=True)
    refs = [oracle_row(x[i], P[i], allow[i] if P[i].get("masked") else None) for i in range(B)]
    errs = compare(x, P, _run_padded(x, P, bits.view(np.int32)), refs=refs)
    assert not errs, "\n".join(errs[:20])


@pytest.mark.parametrize("V", [4096, 8193, 50257, 128256])
def test_infinite_temperature(V):
    """y / inf is 0 of a finite y and NaN of an infinite one, wherever in the
    row it lies: none, one at either end, in a masked, banned, biased or
    unbanned place; k of every kind of list."""
    rng = np.random.default_rng(V)
    B = 18
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    P = [dict(temperature=float("inf"), top_k=k, top_p=0.9, top_logprobs=5, seed=i)
         for i, k in enumerate([0, 1, 40, 128, 300, 600, V // 5, V - 1] + [40] * (B - 8))]
    allow = np.ones((B, V), bool)
    x[8, V - 1] = -np.inf
    x[9, 0] = -np.inf
    x[10, V // 2] = np.inf
    P[11].update(masked=True)                                         # masked, every id allowed
    P[12].update(masked=True)
    allow[12, V - 2] = False
    P[13].update(ban=[V // 3])
    P[14].update(bias=[(V // 3, -np.inf)], top_k=0)
    x[15, 7] = np.inf
    P[15].update(bias=[(7, -np.inf)])                                 # inf - inf
    P[16].update(counts=[(int(t), 2) for t in rng.choice(V, 300, replace=False)], repeat=1.2)
    x[17] = -1.0
    bits = np.zeros((B, (V + 31) // 32), np.uint32)
    for i in range(B):
        bits[i] = np.packbits(np.pad(allow[i], (0, -V % 32)), bitorder="little").view(np.uint32)
    print(f"[case] T = inf V={V}", flush=True)
    refs = [oracle_row(x[i], P[i], allow[i] if P[i].get("masked") else None) for i in range(B)]
    errs = compare(x, P, _run_padded(x, P, bits.view(np.int32)), refs=refs)
    assert not errs, "\n".join(errs[:20])
