"""Softmax over ragged rows on both sides of the size up to which the result is left in the caches."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("heads,s,dtype", [(32, 1915, torch.float16), (32, 1917, torch.float16), (30, 1979, torch.bfloat16)])
def test_causal_rows(hip, heads, s, dtype):
    x = torch.empty((heads, s, s), dtype=dtype, device="cuda").normal_(0, 8)
    out = torch.full_like(x, float("nan"))
    torch.cuda.synchronize()
    hip.call("mh_softmax_causal", None, x.data_ptr(), out.data_ptr(), heads, s, s, 0, 1.0, 0 if dtype == torch.float16 else 1)
    torch.cuda.synchronize()
    mask = torch.full((s, s), float("-inf"), device="cuda").triu(1)
    # half a step of the result (relative, and of its smallest numbers) behind 32-bit exponentials and sums of 2000 terms
    step = (2.0 ** -11 if dtype == torch.float16 else 2.0 ** -8) + 2.0 ** -18
    for h in range(heads):
        want = torch.softmax(x[h].float() + mask, -1)
        assert ((out[h].float() - want).abs() <= step * want + 2.0 ** -25).all(), h
        assert (out[h].triu(1) == 0).all()


@pytest.mark.parametrize("dtype", [torch.float16, torch.bfloat16])
@pytest.mark.parametrize("heads,s", [(20, 420), (21, 420), (35, 604), (34, 604), (82, 340), (83, 340), (12, 766), (12, 770), (180, 149), (180, 151)])
def test_results_that_are_flushed(hip, heads, s, dtype):
    """Both sides of the sizes, numbers of rows and row lengths that keep the hint."""
    test_causal_rows(hip, heads, s, dtype)
