"""Products of more tiles than CUs (csrc/gptq_gemm_tall.hip): the last pass in K ranges, blocks of 128 and of 256 rows,
ragged in rows and columns, with bias and with SiLU * up, and without room for the ranges' sums."""
import pytest
import torch

pytestmark = pytest.mark.gpu


def _weights(k, n, group, bits, seed):
    g = torch.Generator(device="cuda")
    g.manual_seed(seed)
    qweight = torch.randint(-2 ** 31, 2 ** 31, (k * bits // 32, n), dtype=torch.int32, device="cuda", generator=g)
    qzeros = torch.full((k // group, n * bits // 32), 0x77777777 if bits == 4 else 0x7f7f7f7f, dtype=torch.int32, device="cuda")
    scales = ((0.5 + torch.rand((k // group, n), device="cuda", generator=g)) / (k ** 0.5 * (1 << bits))).half()
    return (qweight, qzeros, scales), g


@pytest.mark.parametrize("m,k,n,bits", [
    (1000, 2688, 5120, 4), (1000, 2688, 5112, 8),   # 320 tiles of 128 rows: 64 of them in four ranges, the last one shorter
    (257, 2688, 13312, 4),                          # 312 tiles, one row in the last block
    (900, 4096, 11264, 4), (900, 4096, 11208, 8),   # 352 tiles of 256 rows: 96 in two ranges
    (1281, 4096, 7680, 4),                          # 360 of them, one row in the last block
])
def test_last_pass_in_ranges(hip, m, k, n, bits):
    group = 128
    weight, g = _weights(k, n, group, bits, m + n)
    x = torch.empty((m, k), dtype=torch.float16, device="cuda").normal_(generator=g)
    bias = torch.empty((n,), dtype=torch.float16, device="cuda").normal_(generator=g)
    w = torch.empty((k, n), dtype=torch.float16, device="cuda")
    args = (m, n, k, group, bits)
    need = hip.call("mh_gptq_workspace_bytes", *args)
    assert need > 0   # the sums of the last pass
    torch.cuda.synchronize()
    hip.call("mh_gptq_dequant", None, *(t.data_ptr() for t in weight), None, w.data_ptr(), n, k, group, bits)
    torch.cuda.synchronize()
    want = x.double() @ w.double()

    def close(got, ref, what):
        # fp16 results: half a step of 2^-11, rounded once; sums in 32 bits add 1e-6
        rel = ((got.double() - ref).norm() / ref.norm()).item()
        assert rel <= 3e-4, (what, rel)
        worst = ((got.double() - ref).abs() / ref.abs().clamp(min=ref.std().item())).max().item()
        assert worst <= 1e-3, (what, worst)

    for nbytes in (need, 0):   # no room: whole tiles, the result the same within the sums' order
        ws = torch.zeros(max(nbytes, 256), dtype=torch.uint8, device="cuda")
        out = torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda")
        torch.cuda.synchronize()
        for _ in range(2):
            hip.call("mh_gptq_matmul", None, x.data_ptr(), *(t.data_ptr() for t in weight), None, out.data_ptr(), *args,
                     ws.data_ptr(), nbytes)
        torch.cuda.synchronize()
        close(out, want, "product")
        biased = torch.full_like(out, float("nan"))
        torch.cuda.synchronize()
        hip.call("mh_gptq_linear", None, x.data_ptr(), *(t.data_ptr() for t in weight), None, bias.data_ptr(),
                 biased.data_ptr(), *args, ws.data_ptr(), nbytes)
        torch.cuda.synchronize()
        assert torch.equal(biased, out + bias)
        if n % 256 == 0:
            act = torch.full((m, n // 2), float("nan"), dtype=torch.float16, device="cuda")
            torch.cuda.synchronize()
            assert hip.call("mh_gptq_silu_pairs_workspace_bytes", *args) == need
            hip.call("mh_gptq_matmul_silu_pairs", None, x.data_ptr(), *(t.data_ptr() for t in weight), act.data_ptr(),
                     *args, ws.data_ptr(), nbytes)
            torch.cuda.synchronize()
            pairs = out.double().reshape(m, n // 256, 2, 128)   # 128 gate and 128 up columns per block
            gate, up = pairs[:, :, 0], pairs[:, :, 1]
            close(act, (gate * torch.sigmoid(gate) * up).reshape(m, n // 2), "silu")


@pytest.mark.parametrize("m,k,n", [(1537, 5120, 5120), (800, 4096, 28672), (1000, 2688, 5120)])
def test_static_entry_serves_prompts(hip, m, k, n):
    """The ranges' sums against the built-in buffer of the entry that takes no workspace: more than it holds (the first two:
    whole tiles, the bits of a call without a workspace) or less (the third: the bits of a call with one)."""
    weight, g = _weights(k, n, 128, 4, m)
    x = torch.empty((m, k), dtype=torch.float16, device="cuda").normal_(generator=g)
    args = (m, n, k, 128, 4)
    need, limit = hip.call("mh_gptq_workspace_bytes", *args), hip.call("mh_gptq_static_scratch_bytes")
    assert (need <= limit) == (m == 1000)
    room = need if need <= limit else 0
    ws = torch.zeros(max(room, 256), dtype=torch.uint8, device="cuda")
    got, want = (torch.full((m, n), float("nan"), dtype=torch.float16, device="cuda") for _ in range(2))
    torch.cuda.synchronize()
    operands = (x.data_ptr(), *(t.data_ptr() for t in weight), None)
    hip.call("mh_gptq_matmul_static", None, *operands, got.data_ptr(), *args)
    hip.call("mh_gptq_matmul", None, *operands, want.data_ptr(), *args, ws.data_ptr(), room)
    torch.cuda.synchronize()
    assert torch.equal(got, want) and bool(torch.isfinite(got).all())
