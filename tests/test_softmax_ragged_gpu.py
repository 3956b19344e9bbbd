"""Softmax over rows that are no whole number of 16-byte pieces (or start between two), plain and causal, for every
number of threads per row, with the last piece on either side of the last visible column."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,s,offset", [(3, 9, 0), (2, 7, 1), (2, 33, 92), (2, 130, 0), (1, 9, 1000), (2, 5, 3065),
                                            (1, 17, 4000), (1, 3, 8188)])
def test_ragged_rows(hip, heads, s, offset):
    from minit_amd.hip.tensor import HIPTensor
    t = s + offset
    x = np.random.default_rng(t).normal(0, 8, size=(heads, s, t)).astype(np.float16)
    d, out = HIPTensor.from_numpy(x), HIPTensor.allocate(x.shape, "float16")
    hip.call("mh_softmax", None, d.data_ptr, out.data_ptr, heads * s, t, 1, 0)
    plain = out.numpy()
    scale = np.float32(0.0883)
    hip.call("mh_softmax_causal", None, d.data_ptr, out.data_ptr, heads, s, t, offset, float(scale), 0)
    causal = out.numpy()
    scores = (x.astype(np.float32) * scale).astype(np.float16).astype(np.float64)
    masked = np.where(np.arange(t)[None, :] - offset > np.arange(s)[:, None], -np.inf, scores)
    for got, logits in ((plain, x.astype(np.float64)), (causal, masked)):
        e = np.exp(logits - logits.max(-1, keepdims=True))
        ref = (e / e.sum(-1, keepdims=True)).astype(np.float16).astype(np.float64)
        # one fp16 step: the fp32 exponential and sum are three orders below it
        assert (np.abs(got.astype(np.float64) - ref) <= np.spacing(ref.astype(np.float16)).astype(np.float64)).all()
    assert (causal[:, np.arange(t)[None, :] - offset > np.arange(s)[:, None]] == 0).all()


@pytest.mark.parametrize("s,t", [(40, 40), (150, 150), (600, 1500), (256, 2048), (64, 5001)])
def test_causal_rows_without_a_sum(hip, s, t):
    """NaN, +inf or nothing but -inf among the visible columns: the whole row is NaN, its masked end included."""
    from minit_amd.hip.tensor import HIPTensor
    x = np.random.default_rng(t).normal(size=(s, t)).astype(np.float16)
    offset = t - s
    x[1, 0], x[2, offset], x[4, :offset + 5] = np.nan, np.inf, -np.inf
    x[6, offset + 7:] = np.nan   # masked: counts nowhere
    d, out = HIPTensor.from_numpy(x), HIPTensor.allocate(x.shape, "float16")
    hip.call("mh_softmax_causal", None, d.data_ptr, out.data_ptr, 1, s, t, offset, 1.0, 0)
    got = out.numpy()
    none = np.isin(np.arange(s), (1, 2, 4))
    assert np.isnan(got[none]).all()
    assert np.isfinite(got[~none]).all() and (got[6, offset + 7:] == 0).all()
