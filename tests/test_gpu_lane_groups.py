"""BTOPK for K <= 64 from group maxima (zs_k_lane_scan, zs_k_btopk_pick): rows
and widths where groups, thresholds and lists can go wrong, against the
oracle's WGSL restatement (ids and values bit for bit)."""
import numpy as np
import pytest
import torch

from oracle import oracle as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [50, 4096, 50257, 81921, 163844])
@pytest.mark.parametrize("K", [1, 5, 64])
def test_btopk_from_group_maxima(V, K):
    from tests.gpu_util import ctx
    from zllm_amd.engine import lane_topk
    rng = np.random.default_rng(V + K)
    x = rng.normal(0, 2, (9, V)).astype(np.float32)
    x[0].sort()                                     # the top entries adjacent
    x[1] = 1.5                                      # every key at the threshold
    x[2] = np.where(rng.random(V) < 0.5, np.float32(0.0), np.float32(-0.0))
    x[3] = -np.inf                                  # fewer candidates than K
    x[3, [0, V // 2, V - 1]] = [1.0, np.nan, 2.0]
    x[4] = np.round(x[4])                           # many ties
    x[5, -3:] = [9.0, 3.2e38, 10.0]                 # the last, partial group; beyond the candidates' range
    x[6, V // 3:V // 3 + 2000] = 20.0               # more equal keys than the lists hold
    x[7, ::2] = np.nan
    x[8] = np.nan
    print(f"[case] btopk group maxima V={V} K={K}", flush=True)
    xs = torch.zeros((9, (V + 3) // 4 * 4), device="cuda")
    xs[:, :V] = torch.from_numpy(x)
    vals, idxs = lane_topk(ctx(64, max(151936, V)), xs[:, :V], K)
    vals, idxs = vals.cpu().numpy(), idxs.cpu().numpy().view(np.uint32)
    for s in range(9):
        ov, oi = O.btopk(x[s], K)
        assert idxs[s].tolist() == oi.tolist(), s
        assert vals[s].tobytes() == ov.tobytes(), s


def test_btopk_of_no_ids():
    """Rows of no ids: refused on the group path before anything is launched
    (its kernels index the maxima of the last group), all sentinels past it."""
    from tests.gpu_util import ctx
    from zllm_amd._lib import lib
    c = ctx()
    x = torch.zeros(4, device="cuda")
    vals, idxs = torch.zeros((2, 65), device="cuda"), torch.zeros((2, 65), dtype=torch.int32, device="cuda")
    call = lambda K: lib().zs_lane_topk(c.h, x.data_ptr(), 2, 0, 0, K, vals.data_ptr(), idxs.data_ptr(), None)
    assert call(64) == -1   # ZS_EINVAL
    torch.cuda.synchronize()
    assert not vals.any() and not idxs.any()
    assert call(65) == 0
    torch.cuda.synchronize()
    assert (idxs == -1).all() and (vals < -2.9e38).all()


@pytest.mark.parametrize("V", [3000, 20000, 128256, 163841])
@pytest.mark.parametrize("K", [1, 40, 64])
def test_btopk_many_groups_or_ids(V, K):
    """Rows where more groups or ids than the lists hold reach the first key
    taken: cut to the first K groups, quads and ids by (key desc, id asc)."""
    from tests.gpu_util import ctx
    from zllm_amd.engine import lane_topk
    rng = np.random.default_rng(V + K)
    n = 10
    x = rng.normal(0, 2, (n, V)).astype(np.float32)
    x[0].sort()
    x[1] = np.sort(x[1])[::-1]
    x[2] = np.round(x[2] * 2) / 2                              # ties within and across groups
    x[3, rng.choice(V, 700, replace=False)] = 11.0             # 700 equal maxima, spread
    x[4, rng.choice(V, 63, replace=False)] = rng.uniform(12, 13, 63).astype(np.float32)
    x[4, V // 5:V // 5 + 1500] = 11.0                          # 63 above a run of equal values
    x[5] = np.sort(x[5])
    x[5, -1500::2] = np.nan                                    # candidates and others in turn
    x[6] = rng.integers(0, 2, V).astype(np.float32)
    x[7] = -np.inf
    x[7, V // 3:V // 3 + 40] = 5.0                             # fewer candidates than K, all equal
    x[8, :600] = np.linspace(20, 30, 600, dtype=np.float32)    # the first groups, ascending
    x[9, -1200:] = 3.0e38                                      # beyond the candidates' range
    x[9, -1200:-100:3] = 2.9e38
    print(f"[case] btopk many V={V} K={K}", flush=True)
    xs = torch.zeros((n, (V + 3) // 4 * 4), device="cuda")
    xs[:, :V] = torch.from_numpy(x)
    vals, idxs = lane_topk(ctx(64, max(151936, V)), xs[:, :V], K)
    vals, idxs = vals.cpu().numpy(), idxs.cpu().numpy().view(np.uint32)
    for s in range(n):
        ov, oi = O.btopk(x[s], K)
        assert idxs[s].tolist() == oi.tolist(), s
        assert vals[s].tobytes() == ov.tobytes(), s
