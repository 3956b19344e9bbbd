"""8-bit weights on the kernel of 64-, 128- and 256-row blocks (csrc/gptq_gemm_tall.hip): every number of row tiles,
ragged row and column tiles, K split over workgroups, every group size of the ring, one-hot rows bit for bit."""
import numpy as np
import pytest
import torch

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


@pytest.mark.parametrize("m,k,n", [
    (16, 1024, 28672), (32, 512, 32768), (33, 512, 20480), (64, 1024, 28672),   # two and four row tiles, whole walks
    (100, 512, 16384), (257, 1024, 28672),                                     # blocks of 128 and of 256 rows
    (900, 4096, 11264), (1000, 2688, 5120),                                    # the last pass in K ranges
    (64, 4096, 4096), (9, 6144, 4096)])                                        # K split: the other kernels' SiLU * up
def test_8bit_silu_pairs(hip, m, k, n):
    """SiLU * up of 8-bit products in the store of the row-block kernel, against the product's own fp16 sums."""
    group, bits = 128, 8
    g = torch.Generator(device="cuda")
    g.manual_seed(m + n)
    qweight = torch.randint(-2 ** 31, 2 ** 31, (k // 4, n), dtype=torch.int32, device="cuda", generator=g)
    qzeros = torch.randint(-2 ** 31, 2 ** 31, (k // group, n // 4), dtype=torch.int32, device="cuda", generator=g)
    scales = ((0.5 + torch.rand((k // group, n), device="cuda", generator=g)) / (k ** 0.5 * 128)).half()
    x = torch.empty((m, k), dtype=torch.float16, device="cuda").normal_(generator=g)
    args = (m, n, k, group, bits)
    room = max(hip.call("mh_gptq_workspace_bytes", *args), hip.call("mh_gptq_silu_pairs_workspace_bytes", *args), 256)
    ws = torch.zeros(room, dtype=torch.uint8, device="cuda")
    w, out, act = (torch.full(s, float("nan"), dtype=torch.float16, device="cuda") for s in ((k, n), (m, n), (m, n // 2)))
    operands = (qweight.data_ptr(), qzeros.data_ptr(), scales.data_ptr())
    torch.cuda.synchronize()
    hip.call("mh_gptq_dequant", None, *operands, None, w.data_ptr(), n, k, group, bits)
    hip.call("mh_gptq_matmul", None, x.data_ptr(), *operands, None, out.data_ptr(), *args, ws.data_ptr(), room)
    hip.call("mh_gptq_matmul_silu_pairs", None, x.data_ptr(), *operands, act.data_ptr(), *args, ws.data_ptr(), room)
    torch.cuda.synchronize()
    want = x.double() @ w.double()
    assert ((out.double() - want).norm() / want.norm()).item() <= 3e-4   # one fp16 rounding, sums in 32 bits
    pairs = want.reshape(m, n // 256, 2, 128)   # 128 gate and 128 up columns per block
    silu = (pairs[:, :, 0] * torch.sigmoid(pairs[:, :, 0]) * pairs[:, :, 1]).reshape(m, n // 2)
    # gate and up rounded to fp16 (2.1e-4 each), silu(gate) changing no faster than 1.1 times gate, two more roundings
    assert ((act.double() - silu).norm() / silu.norm()).item() <= 8e-4
