"""LaneBatcher._streams: the knobs packed as bytes and set field by field are
the same zs_lane_stream, for every value that either way takes, and a value
that ctypes refuses is refused."""
import numpy as np
import pytest

from zllm_amd._lib import LaneStream
from zllm_amd.engine import LaneBatcher, LaneSeq, SamplingParams


def _seq(temp=0.7, top_k=40, top_p=0.95, seed=5, n=3):
    s = LaneSeq(0, SamplingParams(temp, top_k, top_p), seed, 0, 100)
    s.generated = [0] * n
    return s


def _batch(seqs):
    b = LaneBatcher(None)
    for s in seqs:
        b.add(s)
    return bytes(b._streams(len(seqs)))


def _fields(seqs):
    st = (LaneStream * max(len(seqs), 1))()
    for i, s in enumerate(seqs):
        st[i].temp, st[i].top_k, st[i].top_p = s.params.temp, s.params.top_k, s.params.top_p
        st[i].base_seed, st[i].gen_index = s.base_seed & 0xFFFFFFFF, s.gen_index() & 0xFFFFFFFF
    return bytes(st)


@pytest.mark.parametrize("knobs", [
    dict(), dict(temp=0), dict(temp=True), dict(temp=np.float32(0.5)), dict(temp=float("inf")), dict(top_p=1e-45),
    dict(top_k=np.int64(7)), dict(seed=2**40 + 9), dict(seed=-3), dict(n=0),
    # refused by a struct code
    dict(temp=1e39), dict(temp=-1e39), dict(top_p=np.float64(1e300)), dict(top_k=-1), dict(top_k=2**32 + 5), dict(top_k=2**70),
])
def test_same_either_way(knobs):
    seqs = [_seq(), _seq(**knobs), _seq(temp=1.1, top_k=0, seed=77, n=9)]
    assert _batch(seqs) == _fields(seqs)


def test_nan_and_no_stream():
    seqs = [_seq(temp=float("nan"))]
    assert np.isnan(LaneStream.from_buffer_copy(_batch(seqs)).temp)
    assert _batch([]) == _fields([]) == bytes(20)


@pytest.mark.parametrize("knobs", [dict(top_k=1.5), dict(top_k="5"), dict(temp=None), dict(top_p="x"), dict(temp=10**400)])
def test_refused(knobs):
    with pytest.raises((TypeError, OverflowError)):
        _batch([_seq(), _seq(**knobs)])
