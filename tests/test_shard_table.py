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
