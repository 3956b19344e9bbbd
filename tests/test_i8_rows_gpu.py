"""GPU parity of the W8A8 product on small tiles with K split over the waves of a workgroup: integer sums and the
fp16 output bit for bit, at the edges of every tile and of the K walk."""
import numpy as np
import pytest

from oracle import int8 as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k", [
    (1, 1, 64),          # half a step, one wave of eight has work
    (16, 1000, 1088),    # 16 x 16 tiles; 8.5 steps: the half step falls to the first wave again
    (17, 4095, 4096),    # one row in the second row tile, N odd: scalar stores
    (48, 1024, 3008),    # 32 x 16 tiles, the last one half empty; K / 64 odd
    (64, 4100, 4096),    # 32 x 32 tiles, four columns over
    (5, 11008, 576),     # 16 x 64 tiles, fewer steps than waves times stages
    (32, 11004, 4160),   # 32 x 64 tiles, 32.5 steps
    (65, 11008, 1024),   # 64 x 64 tiles, one row over
    (300, 2000, 1088),   # 64 x 64 tiles, ragged in rows, columns and K
])
@pytest.mark.parametrize("want_acc", [True, False])
def test_i8_gemm_small_tiles_bit_exact(hip, m, n, k, want_acc):
    from minit_amd import synthetic
    from minit_amd.hip.tensor import HIPTensor
    a, w, a_scale, w_scale = synthetic.int8_operands(f"i8-rows-{m}-{n}-{k}", m, n, k)
    held = [HIPTensor.from_numpy(t) for t in (a, w, a_scale, w_scale)]
    out = HIPTensor.allocate((m, n), "float16")
    acc = HIPTensor.allocate((m, n), "int32") if want_acc else None
    hip.call("mh_i8_gemm", None, *(t.data_ptr for t in held), out.data_ptr, acc.data_ptr if acc else None, m, n, k)
    ref_out, ref_acc = O.gemm(a, w, a_scale, w_scale)
    if acc:
        np.testing.assert_array_equal(acc.numpy(), ref_acc)
    np.testing.assert_array_equal(out.numpy().view(np.uint16), ref_out.view(np.uint16))
