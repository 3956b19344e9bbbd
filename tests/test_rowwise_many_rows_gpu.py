"""Row-wise kernels over more rows than one launch has threads for: 16 threads per short row are more than 2^32 from 2^28
rows on."""
import pytest
import torch

pytestmark = pytest.mark.gpu

ROWS = (1 << 28) + 5
SAMPLES = [slice(r, r + (1 << 16)) for r in (0, 1 << 16, 1 << 27, ROWS - (1 << 16))]


def _input(cols):
    x = torch.empty((ROWS, cols), dtype=torch.float16, device="cuda").normal_()
    torch.cuda.synchronize()
    return x


@pytest.mark.parametrize("cols", [9, 8])   # rows that start anywhere, rows of whole 16-byte pieces
def test_softmax(hip, cols):
    x = _input(cols)
    out = torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    hip.call("mh_softmax", None, x.data_ptr(), out.data_ptr(), ROWS, cols, 1, 0)
    torch.cuda.synchronize()
    for s in SAMPLES:
        # probabilities up to 1: one fp16 rounding
        assert ((out[s].double() - x[s].double().softmax(-1)).abs() <= 2.0 ** -11).all(), s
    assert not torch.isnan(out[:, 0]).any()


def test_rms_norm(hip):
    x = _input(8)
    w, out = torch.ones(8, dtype=torch.float16, device="cuda"), torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    hip.call("mh_rms_norm", None, x.data_ptr(), w.data_ptr(), out.data_ptr(), ROWS, 8, 1, 1e-5, 0)
    torch.cuda.synchronize()
    for s in SAMPLES:
        v = x[s].double()
        want = v / (v.square().mean(-1, keepdim=True) + 1e-5).sqrt()
        assert ((out[s].double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -24).all(), s   # one fp16 rounding
    assert not torch.isnan(out[:, 0]).any()


@pytest.mark.parametrize("what", ["mh_sum", "mh_max"])
def test_reduction(hip, what):
    x = _input(8)
    out = torch.full((ROWS,), float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    hip.call(what, None, x.data_ptr(), out.data_ptr(), ROWS, 8, 1, 0)
    torch.cuda.synchronize()
    for s in SAMPLES:
        v = x[s].double()
        want = v.sum(-1) if what == "mh_sum" else v.amax(-1)
        # one fp16 rounding of sums that are exact to 2^-20 in 32 bits
        assert ((out[s].double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -20).all(), s
    assert not torch.isnan(out).any()
