"""The row kernel's candidate lists at thresholds and sizes where they can go
wrong, compared with the oracle (tokens and top ids bit for bit)."""
import numpy as np
import pytest

from tests.gpu_util import compare, run_gpu

pytestmark = pytest.mark.gpu


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
