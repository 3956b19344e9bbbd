"""The workspace of a quantized product by operators is large enough for what the library takes at the time of the call."""
import random

from minit_amd import lib
from minit_amd.hip import memory

NAME = "mh_gptq_workspace_bytes"
LEAST = 64 << 20   # of the shared workspace


def test_the_switch_read_at_every_call(monkeypatch):
    """The size is kept from the first call of a shape, whatever MH_GEMM_SMALL_KW is set to later."""
    lib.cdll()
    asked, differ = [], 0
    monkeypatch.setattr(memory, "workspace", asked.append)
    rng = random.Random(71)
    shapes = [(32, 256 * tiles, 16384, 128, bits) for tiles in (1, 64, 128, 192, 255, 256, 257) for bits in (4, 8)]
    shapes += [(rng.randint(1, 64), 32 * rng.randint(8, 1 << rng.randint(4, 14)), 256 * rng.randint(1, 112),
                rng.choice((32, 64, 128, 256)), rng.choice((4, 8))) for _ in range(5000)]
    for shape in shapes:
        needed = []
        for setting in ("", "1", "2"):
            monkeypatch.setenv("MH_GEMM_SMALL_KW", setting)
            needed.append(lib.call(NAME, *shape))
            memory.product_workspace(*shape)
            assert max(asked.pop(), LEAST) >= needed[-1], shape
        if len(set(needed)) > 1:
            differ += 1
            assert max(needed) < 20e6, shape
    assert differ > 100
