"""A verification of more workgroups than one launch takes beside a sampler, and
of as many as decide in front of the residual pass and more: every row against
the oracle, the last launch's rows and a last launch that is not full included."""
import numpy as np
import pytest
import torch

from oracle import oracle as O
from zllm_amd.engine import Context, verify_drafts

pytestmark = pytest.mark.gpu


# 33 positions of one chunk a row (24576 workgroups a launch: 744 rows of one): one full launch, two, three
@pytest.mark.parametrize("B", [744, 745, 1500])
def test_rows_of_every_launch(B):
    print(f"[case] spec parts B={B}", flush=True)
    k, V, ld = 16, 37, 40
    rng = np.random.default_rng(B)
    target = rng.normal(0, 2.0, (B, k + 1, ld)).astype(np.float32)
    draft = (target[:, :k] + rng.normal(0, 0.3, (B, k, ld))).astype(np.float32)
    ids = rng.integers(0, V, (B, k)).astype(np.uint32)
    sure = rng.random((B, k)) < 0.9
    ids = np.where(sure, np.argmax(draft[:, :, :V], axis=2), ids).astype(np.uint32)
    temp = np.where(np.arange(B) % 3 == 0, 0.0, 0.8).astype(np.float32)
    seeds = np.arange(B, dtype=np.uint64) + 5
    ctr = np.full(B, 2, np.uint64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    c = Context(max_rows=B, max_vocab=64)
    acc, nxt = verify_drafts(c, t(target)[:, :, :V], t(ids.view(np.int32)), t(temp), t(seeds.view(np.int64)),
                             t(ctr.view(np.int64)), t(draft)[:, :, :V])
    acc, nxt = acc.cpu().numpy(), nxt.cpu().numpy().view(np.uint32)
    c.close()
    for b in range(B):
        want = O.spec_verify(target[b, :, :V], draft[b, :, :V], ids[b].tolist(), float(temp[b]), int(seeds[b]), int(ctr[b]))
        assert (int(acc[b]), int(nxt[b])) == want, (b, (acc[b], nxt[b]), want)


@pytest.mark.parametrize("B", [744, 745, 1500])
def test_rows_of_every_launch_beside_a_sampler(B):
    """The same calls on another stream than the context's sampler: there the
    chunk pass goes in launches of at most 24576 workgroups."""
    from zllm_amd.engine import BatchSampler
    from tests.gpu_util import make_rows
    print(f"[case] spec parts beside B={B}", flush=True)
    c = Context(max_rows=B, max_vocab=64)
    x = torch.randn((4, 40), device="cuda")
    bs = BatchSampler(c)
    bs.run(x, bs.pack(x, make_rows([dict(seed=i) for i in range(4)])))
    other = torch.cuda.Stream()
    other.wait_stream(torch.cuda.current_stream())
    with torch.cuda.stream(other):
        _verify_against_oracle(c, B, 16, 37, 40)
    c.close()


# one chunk a row: 1024 workgroups decide in front of the residual pass, 1025 before it
@pytest.mark.parametrize("B,V", [(1024, 37), (1025, 37), (512, 8193), (513, 8193), (2049, 37)])
@pytest.mark.parametrize("sampled", [True, False])
def test_decision_in_front_and_alone(B, V, sampled):
    print(f"[case] spec decision B={B} V={V} sampled={sampled}", flush=True)
    c = Context(max_rows=B, max_vocab=V)
    _verify_against_oracle(c, B, 2, V, (V + 3) // 4 * 4, sampled)
    c.close()


def _verify_against_oracle(c, B, k, V, ld, sampled=True):
    rng = np.random.default_rng(B + V)
    target = rng.normal(0, 2.0, (B, k + 1, ld)).astype(np.float32)
    draft = (target[:, :k] + rng.normal(0, 0.3, (B, k, ld))).astype(np.float32)
    ids = rng.integers(0, V, (B, k)).astype(np.uint32)
    sure = rng.random((B, k)) < 0.9
    ids = np.where(sure, np.argmax(draft[:, :, :V], axis=2), ids).astype(np.uint32)
    temp = np.where(np.arange(B) % 3 == 0, 0.0, 0.8).astype(np.float32)
    target[B // 2, 0, 3] = np.nan   # verified greedily
    seeds, ctr = np.arange(B, dtype=np.uint64) + 5, np.full(B, 2, np.uint64)
    t = lambda a: torch.from_numpy(np.ascontiguousarray(a)).cuda()
    acc, nxt = verify_drafts(c, t(target)[:, :, :V], t(ids.view(np.int32)), t(temp), t(seeds.view(np.int64)),
                             t(ctr.view(np.int64)), t(draft)[:, :, :V] if sampled else None)
    acc, nxt = acc.cpu().numpy(), nxt.cpu().numpy().view(np.uint32)
    for b in range(B):
        want = O.spec_verify(target[b, :, :V], draft[b, :, :V] if sampled else None, ids[b].tolist(), float(temp[b]),
                             int(seeds[b]), int(ctr[b]))
        assert (int(acc[b]), int(nxt[b])) == want, (b, (acc[b], nxt[b]), want)
