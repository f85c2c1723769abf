"""Which shards the one-launch gather takes (a kernel dereferences them): complete, on the own shard's device, on 16 bytes."""
import types

import pytest

from triton_dist import _lib


def shard(address, device=0):
    return types.SimpleNamespace(data_ptr=lambda: address, get_device=lambda: device)   # (-1: host memory)


@pytest.mark.parametrize("peers,taken", [
    ({0: shard(0x2000), 2: shard(0x3000)}, True),
    ({0: shard(0x2000), 2: shard(0x3000, 1)}, False),   # another GPU: the copies' business
    ({0: shard(0x2000), 2: shard(0x3000, -1)}, False),
    ({0: shard(0x2000), 2: shard(0x3008)}, False),
    ({0: shard(0x2000)}, False),
])
def test_shards_a_kernel_may_read(peers, taken):
    table = _lib.shard_table(shard(0x1000), peers, 1, 3)
    assert (table is not None) == taken
    assert not taken or list(table) == [0x2000, 0x1000, 0x3000]


def test_own_shard_off_16_bytes_and_too_many_ranks():
    assert _lib.shard_table(shard(0x1004), {1: shard(0x2000)}, 0, 2) is None
    n = _lib.GATHER_MAX_RANKS + 1
    assert _lib.shard_table(shard(0x1000), {r: shard(0x1000 * (r + 1)) for r in range(1, n)}, 0, n) is None


@pytest.mark.parametrize("addresses,rows,row_bytes,taken", [
    ([0x1000, 0x2000], 16, 64, True),
    ([1 << 33, (1 << 33) + (1 << 32) - 65536], 16, 64, True),
    ([1 << 33, (1 << 33) + (1 << 32) - 4096], 16, 64, False),   # the last shard's end is out of 32 bits' reach
    ([1 << 33, 1 << 34], 16, 64, False),
    ([0x1000 * (r + 1) for r in range(17)], 16, 64, False),
    ([1 << 20, 1 << 21], 46341, 16, False),                     # 2 * 46341^2 >= 2^32: the division by multiplication ends there
    ([1 << 20, 1 << 21], 46340, 16, True),
    ([1 << 20, 1 << 21], 1, 64, False),                         # 2^32 / 1 is no 32-bit factor
])
def test_shards_read_where_they_lie(addresses, rows, row_bytes, taken):
    assert _lib.shards_in_reach(addresses, rows, row_bytes) == taken


@pytest.mark.parametrize("rows,world", [(2, 16), (3, 16), (50, 4), (2048, 8), (4095, 16), (16383, 16), (46340, 2)])
def test_division_by_a_shards_rows(rows, world):
    """The kernel divides by the high word of a product: exact for every row it may meet."""
    magic = ((1 << 32) + rows - 1) // rows
    assert world * rows * rows < 1 << 32 and magic < 1 << 32
    for shard in range(world):
        for row in (shard * rows, shard * rows + rows - 1, shard * rows + rows // 2):
            assert (row * magic) >> 32 == row // rows
