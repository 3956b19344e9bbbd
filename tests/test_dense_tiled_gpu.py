"""The tiled dense fp16 product (csrc/f16_matmul_tiled.hip) where it can go wrong: lengths of K around its rounds of
64 and its 16-byte pieces, rows that start on odd 2-byte boundaries, ragged tiles of every height (asked for and
asserted), batches whose matrices lie back to back (what follows a row must not leak into it), against the
float64 product; and the one thread per output below eight k."""
import numpy as np
import pytest
import torch

from helpers import assert_fp16_close

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("batch,m,n,k", [
    (1, 1, 1, 8), (2, 5, 7, 9), (3, 33, 129, 63),          # shorter than a round: the remainder alone
    (2, 32, 128, 65), (2, 31, 130, 71), (1, 64, 127, 127),  # one round and 1, 7, 63 elements
    (2, 65, 129, 128), (3, 128, 256, 192), (1, 129, 5, 193), (32, 1500, 100, 130), (2, 96, 130, 200), (3, 97, 129, 129),  # two and three rounds, odd rows
    (2, 200, 300, 1001), (4, 257, 128, 1500), (2, 130, 128, 4096),  # the p v of a prompt
    (1, 2100, 4200, 256), (1, 100, 24600, 512)])            # two tiles per CU; one block of rows
def test_tiled_dense_product(hip, batch, m, n, k):
    _check(hip, batch, m, n, k)


@pytest.mark.parametrize("batch,m,n,k,tile", [
    (2, 65, 129, 127, (64, 1)), (3, 33, 129, 63, (64, 1)),      # one stage in LDS
    (4, 257, 128, 1500, (32, 2)), (2, 31, 130, 131, (32, 2)),
    (8, 1245, 120, 131, (64, 2)), (1, 1250, 1500, 1001, (64, 2)),   # row blocks that end 35 and 30 rows early
    (40, 420, 128, 333, (96, 2)), (32, 1500, 100, 130, (96, 2)),
    (16, 1999, 100, 257, (128, 2)), (30, 1000, 128, 193, (128, 2)),
    (1, 5, 7, 1, (0, 0)), (3, 33, 129, 7, (0, 0)),              # below eight k
])
def test_every_height(hip, batch, m, n, k, tile):
    """Whole blocks of rows and a ragged one, several rounds and a remainder of K, odd rows."""
    assert divmod(hip.call("mh_f16_matmul_tile", batch, m, n, k), 1 << 16) == tile
    _check(hip, batch, m, n, k)


def _check(hip, batch, m, n, k):
    from minit_amd.hip.tensor import HIPTensor
    rng = np.random.default_rng(m * 7 + k)
    a = rng.normal(0, 1, size=(batch, m, k)).astype(np.float16)
    b = rng.normal(0, 0.1, size=(batch, n, k)).astype(np.float16)
    if batch > 1:   # a neighbour's infinities stay in its own rows
        a[1, 0, 0] = np.inf
    out = HIPTensor.allocate((batch, m, n), "float16")
    da, db = HIPTensor.from_numpy(a), HIPTensor.from_numpy(b)
    hip.call("mh_f16_matmul_nk_batched", None, da.data_ptr, db.data_ptr, out.data_ptr, batch, m, n, k)
    got = out.numpy()
    for i in range(batch):
        rows = slice(1, None) if i == 1 else slice(None)
        ref = a[i, rows].astype(np.float64) @ b[i].astype(np.float64).T
        assert_fp16_close(got[i, rows], ref, what=f"matrix {i}")


@pytest.mark.parametrize("batch,m", [(1, (1 << 30) + 70), (1500, 11200 * 64 + 3)])
def test_more_tiles_than_a_launch_holds(hip, batch, m):
    """2^24 tiles and a few more, of one matrix and of a batch: several launches."""
    n, k = 1, 8
    a = torch.empty((batch * m, k), dtype=torch.float16, device="cuda").normal_()
    b = torch.empty((batch, n, k), dtype=torch.float16, device="cuda").normal_()
    out = torch.full((batch * m,), float("nan"), dtype=torch.float16, device="cuda")
    torch.cuda.synchronize()
    hip.call("mh_f16_matmul_nk_batched", None, a.data_ptr(), b.data_ptr(), out.data_ptr(), batch, m, n, k)
    torch.cuda.synchronize()
    assert not torch.isnan(out).any()
    last = batch * m
    for r in (0, 1 << 16, last // 2, last - m, last - 40000):
        rows = torch.arange(r, min(r + 40000, last), device="cuda")
        want = (a[rows].double() * b[rows // m, 0].double()).sum(-1)
        # eight products in 32 bits, one fp16 rounding
        assert ((out[rows].double() - want).abs() <= 2.0 ** -11 * want.abs() + 2.0 ** -18).all(), r
