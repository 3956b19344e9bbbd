"""8-bit weights on the kernel of 64-, 128- and 256-row blocks (csrc/gptq_gemm_tall.hip): every number of row tiles,
ragged row and column tiles, K split over workgroups, every group size of the ring, one-hot rows bit for bit."""
import numpy as np
import pytest

from helpers import assert_fp16_close
from oracle import gptq as O
from test_gptq_gpu import _run_linear, _weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,g", [
    (33, 512, 264, 128), (64, 640, 136, 32),        # one block of 64 rows: four rounds (the ring alone), ragged columns
    (65, 512, 264, 128), (128, 4096, 1024, 128),    # blocks of 128 rows: one ragged; K split over workgroups
    (200, 1024, 776, 64), (384, 2048, 520, 256),    # two and three blocks, groups shorter and longer than a round
    (256, 512, 28672, 128), (500, 384 + 128, 14400, 64), (256, 640, 28800, 32),   # blocks of 256 rows
    (9, 6144, 4096, 128), (17, 4096, 4104, 64), (32, 4096, 4096, 256)])           # two row tiles
def test_8bit_row_blocks(hip, m, k, n, g):
    from minit_amd import synthetic
    qweight, qzeros, scales = _weights(k, n, g, 8, seed=91, zero_range=(0, 255))
    scales = (scales.astype(np.float32) / 16).astype(np.float16)
    x = synthetic.activations("tall8", f"x{m}_{k}", (m, k))
    x[m // 2] = 0
    x[m // 2, k - 1] = 1.0
    got = _run_linear(hip, "mh_gptq_matmul", x, qweight, qzeros, scales, g, 8)
    w = O.dequantize_packed(qweight, qzeros, scales, None, 8, g)
    np.testing.assert_array_equal(got[m // 2].view(np.uint16), w[k - 1].view(np.uint16))
    assert_fp16_close(got, x.astype(np.float64) @ w.astype(np.float64), what=f"8-bit rows {m}x{k}x{n} g{g}")
