"""The free list behind the tensors: bounded, the sizes used last kept, close sizes sharing blocks."""
import pytest

from minit_amd.hip import memory


@pytest.fixture
def device(monkeypatch):
    """mh_malloc / mh_free on a host that counts: live pointers and their sizes."""
    live, calls = {}, []

    def call(name, *args):
        calls.append(name)
        if name == "mh_malloc":
            pointer = 0x1000 * len(calls)
            args[0]._obj.value = pointer
            live[pointer] = args[1]
        elif name == "mh_free":
            del live[args[0]]   # a block given back twice is an error
        return 0

    monkeypatch.setattr(memory.lib, "call", call)
    monkeypatch.setattr(memory, "_POOL", type(memory._POOL)())
    monkeypatch.setattr(memory, "_POOL_BYTES", 0)
    monkeypatch.setattr(memory, "_LENT", {}, raising=False)
    return live, calls


@pytest.mark.parametrize("size", [0, 1, 256, 257, 1 << 20, (1 << 20) + 1, 3 << 20, (1 << 28) - 5, (1 << 28) + 5,
                                  1 << 30, (1 << 30) + 1])
def test_block_sizes(size):
    block = memory._round(size)
    assert block >= max(size, 256) and block % 256 == 0
    assert memory._round(block) == block                 # release finds the block allocate gave
    assert block - size <= max(256, size // 8 if 1 << 20 < size <= 1 << 30 else 0)


def test_sizes_used_last_stay(device):
    live, calls = device
    block = 256 << 20
    old = [memory.allocate(block) for _ in range(14)]
    for p in old:
        memory.release(p, block)
    new_size = 500 << 20
    for _ in range(3):   # the pool is nearly full of another size: the second pass on has its blocks
        pair = [memory.allocate(new_size) for _ in range(2)]
        for p in pair:
            memory.release(p, new_size)
    assert calls.count("mh_malloc") == 16
    assert memory._POOL_BYTES == sum(live.values()) <= memory._POOL_LIMIT
    memory.empty_cache()
    assert not live and memory._POOL_BYTES == 0


def test_blocks_above_the_limit_are_given_back(device):
    live, calls = device
    memory.release(memory.allocate(5 << 30), 5 << 30)
    assert not live and memory._POOL_BYTES == 0


@pytest.mark.parametrize("size", [1, 300, 5120 * 13696, 5120 * 13824 // 2, (1 << 20) + 1, 200_000_001])
def test_new_blocks_are_no_larger_than_asked_for(device, size):
    """Weights and caches stay: 8-bit 5120 x 13696 takes its 70.1 MB and not the 75.5 of a rounder size."""
    live, _ = device
    memory.allocate(size)
    assert sum(live.values()) <= max(256, size + 255)


def test_close_sizes_share_blocks(device):
    live, calls = device
    large, small = 100 << 20, 90 << 20   # within an eighth
    block = memory.allocate(large)
    memory.release(block, large)
    assert memory.allocate(small) == block and calls.count("mh_malloc") == 1 and memory._POOL_BYTES == 0
    memory.release(block, small)
    assert memory._POOL_BYTES == large == sum(live.values())   # a block keeps its size
    other = memory.allocate(80 << 20)                          # more than an eighth less
    assert other != block and memory.allocate(large) == block
    memory.release(block, large)
    memory.release(other, 80 << 20)
    memory.empty_cache()
    assert not live and memory._POOL_BYTES == 0


def test_small_sizes_do_not_share(device):
    _, calls = device
    memory.release(memory.allocate(1 << 20), 1 << 20)
    memory.allocate((1 << 20) - 4096)
    assert calls.count("mh_malloc") == 2


def test_a_tensor_dies_while_a_block_is_put_back(device, monkeypatch):
    """The collector runs inside release(), where the list of a new size has been looked up and not yet stored."""
    live, _ = device
    size = 1 << 16
    blocks = [memory.allocate(size) for _ in range(2)]

    class Pool(type(memory._POOL)):
        dying = [blocks[1]]

        def _die(self):
            while self.dying:
                memory.release(self.dying.pop(), size)

        def get(self, key, default=None):
            value = super().get(key, default)
            self._die()
            return value

        def setdefault(self, key, default=None):
            self._die()
            return super().setdefault(key, default)

    monkeypatch.setattr(memory, "_POOL", Pool())
    memory.release(blocks[0], size)
    assert memory._POOL_BYTES == 2 * size
    assert sorted(p for bucket in memory._POOL.values() for p in bucket) == sorted(blocks)


def test_a_tensor_dies_while_blocks_are_given_back(device, monkeypatch):
    """The collector runs inside hipFree's call, in eviction and in empty_cache()."""
    live, _ = device
    call, dying = memory.lib.call, []
    size = 1 << 30
    blocks = [memory.allocate(size) for _ in range(6)]

    def call_and_collect(name, *args):
        result = call(name, *args)
        if name == "mh_free" and dying:
            memory.release(dying.pop(), size)
        return result

    monkeypatch.setattr(memory.lib, "call", call_and_collect)
    for block in blocks[:4]:
        memory.release(block, size)
    dying.append(blocks[5])
    memory.release(blocks[4], size)   # evicts one, and another for the block that dies meanwhile
    assert not dying and memory._POOL_BYTES == sum(live.values()) <= memory._POOL_LIMIT
    assert sum(len(bucket) for bucket in memory._POOL.values()) == len(live) == 4
    dying.append(memory.allocate(size))
    memory.empty_cache()
    assert not live and memory._POOL_BYTES == 0
