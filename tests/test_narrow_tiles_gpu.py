"""GPU parity of the column-owner kernel's tiles of 16 columns and of its rings without refills, at the lengths
of K where the number of waves and the ring change and at the widths where the order of the tiles does."""
import numpy as np
import pytest

from helpers import assert_fp16_close
from oracle import gptq as O
from test_gptq_gpu import _run_linear, _run_with_bias, _weights

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("m,k,n,g,bits", [
    # K: one ring on 8 waves, on 16, refills, 16 waves with 16 steps, refills again
    (1, 2048, 32, 128, 4), (1, 2304, 96, 128, 4), (2, 4096, 288, 128, 4), (1, 4352, 288, 128, 4), (1, 6144, 256, 128, 4),
    (3, 6400, 288, 128, 4), (8, 8192, 544, 128, 4), (1, 8448, 512, 128, 4), (4, 14336, 2080, 128, 4), (2, 20480, 3104, 128, 4), (5, 10240, 544, 64, 4), (5, 10496, 544, 64, 4), (8, 14336, 3104, 128, 4),
    # one tile of 16 columns per CU, and the first width with tiles of 32 (without refills too)
    (1, 4096, 4096, 128, 4), (8, 2048, 4096, 64, 4), (1, 4096, 4128, 128, 4), (7, 2048, 4128, 128, 4), (8, 3328, 8192, 256, 4),
    # 8 bit, group sizes
    (1, 2048, 96, 32, 8), (5, 4096, 288, 64, 8), (8, 4096, 288, 256, 8), (2, 8192, 288, 32, 8), (8, 8192, 2080, 256, 8),
    (1, 6400, 544, 128, 8), (1, 4096, 4128, 64, 8), (8, 8192, 96, 32, 4), (1, 8192, 96, 256, 4),
    # more rows than 16 waves hold
    (9, 2048, 288, 128, 4), (16, 4096, 4096, 128, 4), (17, 1024, 288, 64, 4), (32, 768, 96, 128, 8),
    # where 17 to 32 rows stay here and where they leave, both widths
    (17, 4096, 4128, 128, 4), (32, 4096, 4096, 64, 8), (20, 6144, 2080, 128, 4), (32, 6400, 544, 128, 4), (31, 4352, 4128, 128, 4),
    (32, 4352, 544, 128, 8),
    # more tiles than CUs: both ring lengths, the widths and lengths where they end, one more each
    (1, 2048, 11008, 128, 4), (8, 1024, 8224, 128, 4), (3, 256, 32768, 128, 4), (1, 2048, 32800, 128, 4), (8, 4096, 14336, 128, 4),
    (2, 4096, 16384, 64, 4), (1, 3840, 24576, 128, 4), (5, 4096, 16416, 128, 4), (4, 3584, 16416, 128, 4), (1, 4352, 14336, 128, 4),
    (8, 2048, 8224, 128, 8), (1, 768, 16384, 32, 8), (1, 768, 16416, 32, 8), (1, 1024, 24576, 256, 8), (1, 2304, 11008, 128, 8), (9, 2048, 11008, 128, 4),
    # 9 to 16 rows: the longest K of either width, and the first that leaves
    (9, 6144, 544, 128, 8), (16, 6144, 2080, 64, 8), (16, 6400, 1056, 128, 8), (9, 8192, 1024, 128, 8), (16, 8192, 544, 128, 4), (9, 8448, 544, 32, 4),
])
def test_products(hip, m, k, n, g, bits):
    from minit_amd import synthetic
    qweight, qzeros, scales = _weights(k, n, g, bits, seed=61, zero_range=(0, (1 << bits) - 1))
    x = synthetic.activations("narrow", f"x{m}_{k}", (m, k))
    got = _run_linear(hip, "mh_gptq_matmul", x, qweight, qzeros, scales, g, bits)
    assert_fp16_close(got, O.matmul_f64(x, qweight, qzeros, scales, None, bits, g), what=f"{m}x{k}x{n}")
    # rows of W picked bit for bit, the ends of K among them
    rows = np.random.default_rng(62).choice(k, size=m, replace=False)
    rows[0], rows[-1] = (k - 1, 0) if m > 1 else (k - 1, k - 1)
    onehot = np.zeros((m, k), dtype=np.float16)
    onehot[np.arange(m), rows] = 1.0
    w = O.dequantize_packed(qweight, qzeros, scales, None, bits, g)
    got = _run_linear(hip, "mh_gptq_matmul", onehot, qweight, qzeros, scales, g, bits)
    np.testing.assert_array_equal(got.view(np.uint16), w[rows].view(np.uint16))
    bias = np.random.default_rng(63).normal(0, 1, n).astype(np.float16)
    got = _run_with_bias(hip, onehot, qweight, qzeros, scales, bias, g, bits)[0]
    np.testing.assert_array_equal(got.view(np.uint16), (w[rows] + bias).view(np.uint16))


@pytest.mark.parametrize("m,k,n,g,bits", [
    # the longest K of groups of 32 and 64, and the first that leaves
    (3, 18432, 3104, 32, 4), (4, 18688, 3104, 32, 4), (1, 20480, 3104, 32, 4), (4, 20736, 3104, 64, 4), (2, 20736, 3616, 32, 4),
    (5, 12288, 3104, 32, 4), (8, 12544, 3104, 32, 4), (6, 12544, 3616, 32, 4), (1, 3840, 16416, 64, 4), (4, 4096, 16416, 32, 4),
    # 17 to 32 rows: both sides of the lines
    (20, 2048, 4128, 32, 4), (32, 2304, 6144, 32, 4), (32, 3328, 6176, 32, 4), (17, 3584, 6144, 32, 4),
    (32, 6144, 1856, 64, 4), (17, 6144, 1888, 64, 4), (24, 6144, 2080, 128, 4), (25, 6144, 2080, 128, 4), (24, 4352, 2080, 256, 4),
])
def test_products_at_the_lines_of_small_groups(hip, m, k, n, g, bits):
    test_products(hip, m, k, n, g, bits)
