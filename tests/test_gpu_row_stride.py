"""Contexts whose max_vocab is the rows' width and no multiple of 4: a row's
scratch may not run into the next row's. Every row without a cut (its kept list
is the whole row) and with most of its mass on the first three ids, so that a
lost head moves the drawn token; tokens against the oracle, on several passes."""
import numpy as np
import pytest
import torch

from tests.gpu_util import compare, make_rows, oracle_row
from zllm_amd.engine import BatchSampler, Context

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("V", [5001, 5002, 5003, 71305])
def test_rows_keep_their_heads(V):
    print(f"[case] row stride V={V}", flush=True)
    B = 48
    rng = np.random.default_rng(V)
    x = rng.normal(0, 0.5, (B, V)).astype(np.float32)
    x[:, :3] = np.log(V / 4.0)
    params = [dict(temperature=1.0, top_p=1.0 if i % 3 else 0.95, seed=i, counter=i) for i in range(B)]
    refs = [oracle_row(x[i], params[i]) for i in range(B)]
    c = Context(max_rows=B, max_vocab=V)
    xs = torch.zeros((B, (V + 3) // 4 * 4), device="cuda")
    xs[:, :V] = torch.from_numpy(x)
    bs = BatchSampler(c)
    bufs = bs.pack(xs[:, :V], make_rows(params))
    for _ in range(4):
        out = bs.run(xs[:, :V], bufs)
        torch.cuda.synchronize()
        errs = compare(x, params, {k: v.cpu().numpy() for k, v in out.items()}, refs=refs)
        assert not errs, "\n".join(errs[:20])
    c.close()
