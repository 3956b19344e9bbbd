"""The decode loop over the column-owner kernel's tiles of 16 columns: residual add with its sums of squares, norm
prologue, RoPE and cache append on rings of 16 waves and on refills, with biases, against the oracle's decode step.

Up to 8 rows (at 16 the longer K leave for other kernels) the narrow products are
  4096 wide: o one ring on 16 waves, down refills; q|k|v is 6144 wide, in tiles of 32 columns that read pieces of 16
  2304 wide: q|k|v one ring on 16 waves, o one ring on 8, down 16 waves with 16 steps each
  8192 wide: q|k|v 16 waves with 16 steps each; o in tiles of 32 columns
  5120 wide: q|k|v refills
"""
import numpy as np
import pytest

from test_decode_biased_gpu import _model, _run_and_check

pytestmark = pytest.mark.gpu

COMMON = dict(n_layers=2, head_dim=128, vocab=256, rope_theta=5e5, rms_eps=1e-5)
CONFIGS = [dict(COMMON, hidden=4096, n_q_heads=32, n_kv_heads=8, ffn=14336, group_size=128, bits=4),
           dict(COMMON, hidden=2304, n_q_heads=16, n_kv_heads=4, ffn=6400, group_size=128, bits=4),
           dict(COMMON, hidden=2304, n_q_heads=16, n_kv_heads=4, ffn=6400, group_size=32, bits=8),
           dict(COMMON, hidden=8192, n_q_heads=16, n_kv_heads=4, ffn=2048, group_size=64, bits=4),
           dict(COMMON, hidden=8192, n_q_heads=16, n_kv_heads=4, ffn=2048, group_size=256, bits=8),
           dict(COMMON, hidden=5120, n_q_heads=16, n_kv_heads=4, ffn=512, group_size=128, bits=4)]

GAIN = [0.25, 1, 2, 0.375, 2, 1]   # on the scales of o and down


@pytest.fixture(scope="module", params=range(len(CONFIGS)), ids=lambda i: f"{CONFIGS[i]['hidden']}-{CONFIGS[i]['bits']}bit")
def model(request):
    model = _model(CONFIGS[request.param], 160 + request.param, act_order=False)
    # neither so small beside the stream that an error in them is lost, nor so large that everything before them is
    gain = np.float16(GAIN[request.param])
    for layer in model["layers"]:
        for name in ("o", "down"):
            qweight, qzeros, scales, *rest = layer[name]
            layer[name] = (qweight, qzeros, scales * gain, *rest)
    return model


@pytest.mark.parametrize("batch", [1, 3, 8, 16])
def test_one_step(hip, model, batch):
    _run_and_check(model["config"], model, batch)
