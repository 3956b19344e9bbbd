"""GPU parity of the W8A8 product on small tiles with K split over the waves of a workgroup: integer sums and the
fp16 output bit for bit, at the edges of every tile and of the K walk.  The tile is asked for and asserted, so
that a change of the rule that picks it cannot take a kernel out of the test."""
import numpy as np
import pytest
import torch

from oracle import int8 as O

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,n,k,tile", [
    (1, 1, 64, (128, 256)),        # too short for small tiles to win
    (1, 138, 128, (16, 16)),       # one step, one wave of eight has work
    (16, 1000, 1088, (16, 16)),    # 8.5 steps: the half step falls to the first wave again
    (48, 1024, 3008, (16, 16)),    # K / 64 odd
    (5, 11008, 576, (16, 16)),     # fewer steps than waves times stages
    (17, 4095, 4096, (32, 16)),    # one row in the second row tile, N odd: scalar stores
    (21, 2153, 448, (32, 16)),     # 3.5 steps: no refill
    (64, 4096, 4096, (32, 32)),    # eight steps per wave: the ring of two wraps
    (8, 5338, 3328, (32, 32)),     # half a tile of rows, two columns over
    (5, 27970, 9856, (16, 64)),    # 19.25 steps per wave
    (10, 10962, 3392, (16, 64)),   # 26.5 steps
    (64, 4100, 4096, (32, 64)),
    (32, 11004, 4160, (32, 64)),   # 32.5 steps
    (33, 5654, 128, (32, 64)),     # one row in the second row tile, a single step
    (66, 5541, 128, (64, 64)),
    (65, 11008, 1024, (128, 256)),
    (70, 5701, 2112, (64, 64)),    # 16.5 steps, ragged in rows and columns
    (300, 2000, 1088, (64, 64)),   # ragged in rows, columns and K
])
@pytest.mark.parametrize("want_acc", [True, False])
def test_i8_gemm_small_tiles_bit_exact(hip, m, n, k, tile, want_acc):
    from minit_amd import synthetic
    from minit_amd.hip.tensor import HIPTensor
    assert divmod(hip.call("mh_i8_gemm_tile", m, n, k), 1 << 16) == tile
    a, w, a_scale, w_scale = synthetic.int8_operands(f"i8-rows-{m}-{n}-{k}", m, n, k)
    held = [HIPTensor.from_numpy(t) for t in (a, w, a_scale, w_scale)]
    out = HIPTensor.allocate((m, n), "float16")
    acc = HIPTensor.allocate((m, n), "int32") if want_acc else None
    hip.call("mh_i8_gemm", None, *(t.data_ptr for t in held), out.data_ptr, acc.data_ptr if acc else None, m, n, k)
    ref_out, ref_acc = O.gemm(a, w, a_scale, w_scale)
    if acc:
        np.testing.assert_array_equal(acc.numpy(), ref_acc)
    np.testing.assert_array_equal(out.numpy().view(np.uint16), ref_out.view(np.uint16))


def test_more_rows_than_a_launch_of_small_tiles_holds(hip):
    """2^29 rows of one column: 32 x 16 tiles of 256 threads each would be 2^32 threads."""
    m, k = (1 << 29) + 37, 64
    a = torch.randint(-2 ** 31, 2 ** 31, (m, k // 4), dtype=torch.int32, device="cuda").view(torch.int8)
    w = torch.randint(-128, 128, (1, k), dtype=torch.int8, device="cuda")
    acc = torch.full((m,), 1 << 30, dtype=torch.int32, device="cuda")
    torch.cuda.synchronize()
    hip.call("mh_i8_gemm", None, a.data_ptr(), w.data_ptr(), None, None, None, acc.data_ptr(), m, 1, k)
    torch.cuda.synchronize()
    for r in (0, 1 << 20, m // 2, m - (1 << 20)):
        s = slice(r, r + (1 << 20))
        assert torch.equal(acc[s].float(), (a[s].float() * w.float()).sum(-1)), r   # below 2^24: exact
    assert int(acc.max()) < 1 << 30
