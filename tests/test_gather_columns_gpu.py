"""mh_gather_columns on its kernels: four columns per thread (16-bit, whole 16-byte pieces, few elements), a row parked
in LDS (more, up to 64 KiB) and one element per thread; index entries outside the row are clamped into it."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,cols,dtype", [(1, 8, np.float16), (3, 4104, np.float16), (300, 4112, np.float16), (1100, 952, np.float16), (33, 32768, np.float16),
                                             (2, 32776, np.float16), (5, 12, np.float16), (4, 2048, np.float32)])
def test_gather_columns(hip, rows, cols, dtype):
    from minit_amd.hip.tensor import HIPTensor
    rng = np.random.default_rng(cols)
    x = rng.normal(size=(rows, cols)).astype(dtype)
    index = rng.permutation(cols).astype(np.int32)
    index[0], index[-1] = -5, cols + 7
    dx, di, out = HIPTensor.from_numpy(x), HIPTensor.from_numpy(index), HIPTensor.allocate((rows, cols), x.dtype.name)
    hip.call("mh_gather_columns", None, dx.data_ptr, di.data_ptr, out.data_ptr, rows, cols, 0 if dtype == np.float16 else 2)
    np.testing.assert_array_equal(out.numpy(), x[:, np.clip(index, 0, cols - 1)])


@pytest.mark.parametrize("rows,cols", [(33, 512), (7, 4104), (4096, 376), (4097, 376), (4100, 384), ((1 << 24) + 3, 8), (1 << 24, 384)])
def test_gather_many_rows(hip, rows, cols):
    """bfloat16 on every kernel: four columns per thread, the widths and row counts at which a row parked in LDS takes
    over from it and from one element per thread, more rows than a launch of a workgroup each can hold."""
    x = torch.randint(-2 ** 31, 2 ** 31, (rows, cols // 2), dtype=torch.int32, device="cuda").view(torch.float16)
    index = torch.randperm(cols, device="cuda").to(torch.int32)
    out = torch.zeros_like(x)
    torch.cuda.synchronize()
    hip.call("mh_gather_columns", None, x.data_ptr(), index.data_ptr(), out.data_ptr(), rows, cols, 1)
    torch.cuda.synchronize()
    for r in range(0, rows, 1 << 20):   # the bits, compared as integers
        want = x[r:r + (1 << 20)].view(torch.int16)[:, index.long()]
        assert torch.equal(out[r:r + (1 << 20)].view(torch.int16), want), r
