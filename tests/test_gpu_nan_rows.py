"""NaN rows in one batch with masked rows, rows of a wide top-k and greedy
rows, while a verification runs on a second stream. Every pass against the
oracle (tokens and top ids bit for bit, floats within gpu_util.compare's
1e-5) and the same in every pass."""
import numpy as np
import pytest
import torch

from tests.gpu_util import compare, ctx, make_rows, oracle_row

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [4096, 32000, 128256])
def test_nan_rows_beside_others(V):
    from zllm_amd.engine import BatchSampler, Context, verify_drafts
    rng = np.random.default_rng(V)
    B, k = 24, 2
    x = rng.normal(0, 2, (B, V)).astype(np.float32)
    allow = np.ones((B, V), bool)
    P = []
    for i in range(B):
        kind = i % 6
        p = dict(temperature=0.9, top_k=40, top_p=0.95, top_logprobs=5, seed=i)
        if kind == 0:
            x[i, rng.integers(0, V, 1 + i)] = np.nan                 # one NaN and many
        elif kind == 1:
            p.update(masked=True, top_k=0)
            allow[i] = rng.random(V) < 0.5
        elif kind == 2:
            p.update(top_k=min(1500, V // 3))
        elif kind == 3:
            x[i, [3, V // 2, V - 1][i // 6 % 3]] = np.nan            # the first, a middle and the last group
            p.update(temperature=0.0)
        elif kind == 4:
            x[i, 17] = np.inf                                        # inf - inf: NaN in y, not in x~
            p.update(bias=[(17, -np.inf)], top_k=0)
        else:
            x[i, 9] = np.nan                                         # a banned NaN is none
            p.update(ban=[9])
        P.append(p)
    bits = np.zeros((B, (V + 31) // 32), np.uint32)
    for i in range(B):
        bits[i] = np.packbits(np.pad(allow[i], (0, -V % 32)), bitorder="little").view(np.uint32)
    refs = [oracle_row(x[i], P[i], allow[i] if P[i].get("masked") else None) for i in range(B)]
    c, c2 = ctx(64, 151936), Context(0, 64, V)
    xs, ab = torch.from_numpy(x).cuda(), torch.from_numpy(bits.view(np.int32)).cuda()
    bs = BatchSampler(c)
    bufs = bs.pack(xs, make_rows(P))
    target = torch.randn((64, k + 1, V), device="cuda")
    draft, ids = target[:, :k].clone(), target[:, :k].argmax(2).to(torch.int32)
    T, z = torch.ones(64, device="cuda"), torch.zeros(64, dtype=torch.int64, device="cuda")
    other, first = torch.cuda.Stream(), None
    for n in range(3):
        print(f"[case] NaN rows V={V} pass {n}", flush=True)
        other.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(other):
            acc, nxt = verify_drafts(c2, target, ids, T, z, z, draft)
        out = bs.run(xs, bufs, ab)
        torch.cuda.synchronize()
        out = {key: v.cpu().numpy() for key, v in out.items()}
        assert (acc == k).all()   # the draft is the target
        if first is None:
            first = out
            errs = compare(x, P, out, refs=refs)
            assert not errs, "\n".join(errs[:20])
        for key in out:
            assert out[key].tobytes() == first[key].tobytes(), (key, n)
    c2.close()
