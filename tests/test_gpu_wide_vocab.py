"""Rows up to the widest vocabulary a context takes (262144 ids): where the row
kernel's bitmaps, the bias windows and the group maxima share a CU's LDS
differently. Against the oracle (tokens and top ids bit for bit, floats within
gpu_util.compare's 1e-5)."""
import numpy as np
import pytest

from tests.gpu_util import compare
from tests.test_gpu_scan import _case, _run_padded

pytestmark = pytest.mark.gpu


# the last width of one bias window and the first of two (about 181900), two
# between, the last with group maxima and the first without (about 242600), the widest
@pytest.mark.parametrize("V", [180224, 184320, 200019, 240640, 245760, 262144])
def test_widest_rows(V):
    x, P = _case(V)
    rng = np.random.default_rng(V)
    for i, n in ((12, 60), (15, 3000)):
        # biases over the whole row, some ids two and three times, near and far apart in the list
        ids = rng.choice(V, n, replace=False).tolist() + [0, V - 1, V // 2]
        ids += ids[:n // 3] + ids[:5]
        P[i].update(top_k=0, bias=[(int(t), float(b)) for t, b in zip(ids, rng.uniform(-6, 4, len(ids)))])
    # more patches than the list's LDS head holds
    P[6].update(counts=[(int(t), 1) for t in rng.choice(V, 6000, replace=False)], presence=0.5,
                bias=[(5, 1.0), (V - 2, 2.0), (5, -0.5), (V - 2, -0.25)])
    print(f"[case] widest rows V={V}", flush=True)
    errs = compare(x, P, _run_padded(x, P))
    assert not errs, "\n".join(errs[:20])
