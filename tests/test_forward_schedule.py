"""The tile lists of the attention forward with the hand-scheduled loop, on the
host alone: whatever the shape, every (sequence, head, query tile) is launched
exactly once, lists never exceed the table, and the heads that share a kv head
stay on as few XCDs as the partitioning promises (workgroup i runs on XCD i mod
8); tiles whose keys are shared out have every key in one part.  No GPU is
needed: the packing is host code behind test-support exports."""
import ctypes
import random

import pytest

from pluto_amd import capi

NO_ITEM = 0xFFFF
CAPACITY = 1536


@pytest.fixture(scope="module")
def library():
    return capi.lib()


def schedule(library, head_dim, q_rows, kv_rows, start, query_heads, group, sequences, resident):
    items = (ctypes.c_uint16 * CAPACITY)()
    workgroups, slots = ctypes.c_int(-1), ctypes.c_int(-1)
    status = library.pluto_hip_test_forward_schedule(
        head_dim, q_rows, kv_rows, start, query_heads, group, sequences, resident, items, CAPACITY,
        ctypes.byref(workgroups), ctypes.byref(slots))
    return status, workgroups.value, slots.value, list(items)


def tile_rows(head_dim):
    return 256 if head_dim == 128 else 128


def check(library, head_dim, q_rows, query_heads, group, sequences, resident, start=0):
    kv_rows = start + q_rows
    status, workgroups, slots, items = schedule(library, head_dim, q_rows, kv_rows, start,
                                                query_heads, group, sequences, resident)
    assert status == 0
    q_tiles = -(-q_rows // tile_rows(head_dim))
    total = q_tiles * query_heads * sequences
    if workgroups == 0:
        return False      # numbered by workgroup index: nothing to check here
    assert workgroups == resident and 0 < slots and workgroups * slots <= CAPACITY
    seen = {}
    for w in range(workgroups):
        ended = False
        for e in range(slots):
            item = items[w * slots + e]
            if item == NO_ITEM:
                ended = True
                continue
            assert not ended, "an entry after the end of a list"
            assert item < total
            assert item not in seen, "tile %d in the lists of workgroups %d and %d" % (item, seen[item], w)
            seen[item] = w
    assert len(seen) == total, "%d of %d tiles are in no list" % (total - len(seen), total)
    # heads of one (sequence, kv head) run on one XCD when the units divide over the eight,
    # on 8 / units XCDs when there are fewer units than XCDs
    kv_heads = query_heads // group
    kv_units = sequences * kv_heads
    xcds = {}
    for item, w in seen.items():
        column = item // q_tiles
        unit = (column // query_heads) * kv_heads + (column % query_heads) // group
        xcds.setdefault(unit, set()).add(w % 8)
    if kv_units % 8 == 0:
        assert all(len(x) == 1 for x in xcds.values())
    elif 8 % kv_units == 0:
        assert all(len(x) <= 8 // kv_units for x in xcds.values())
        assert len(set().union(*xcds.values())) == 8
    # balance: no list carries more than the mean plus one heaviest tile
    def cost(item):
        t = item % q_tiles
        last = min((t + 1) * tile_rows(head_dim), q_rows) - 1
        return -(-min(kv_rows, start + last + 1) // 64) + 8
    loads = [0] * workgroups
    for item, w in seen.items():
        loads[w] += cost(item)
    heaviest = max(cost(i) for i in seen)
    assert max(loads) <= sum(loads) / workgroups + heaviest
    return True


def test_benchmarked_shapes(library):
    assert check(library, 128, 8192, 24, 6, 1, 256)      # the prefill configuration
    assert check(library, 256, 8192, 24, 6, 1, 256)
    assert check(library, 64, 4096, 12, 1, 4, 512)
    assert check(library, 128, 2301, 6, 3, 1, 256) is False   # fewer tiles than workgroups


def test_every_tile_is_launched_once_whatever_the_shape(library):
    rng = random.Random(5)
    listed = 0
    for _ in range(400):
        head_dim = rng.choice([64, 128, 256])
        group = rng.choice([1, 1, 2, 3, 6, 8])
        query_heads = group * rng.randint(1, 6)
        sequences = rng.randint(1, 5)
        q_rows = rng.choice([rng.randint(1, 3000), rng.randint(3000, 40000)])
        start = rng.choice([0, 0, rng.randint(1, 5000)])
        resident = rng.choice([256, 512, 64, 8, 304, 0, 250])
        listed += bool(check(library, head_dim, q_rows, query_heads, group, sequences, resident, start))
    assert listed > 80    # the sample does exercise the packing


def test_rejections(library):
    items = (ctypes.c_uint16 * 4)()
    w, s = ctypes.c_int(), ctypes.c_int()
    call = library.pluto_hip_test_forward_schedule
    assert call(96, 100, 100, 0, 4, 1, 1, 256, items, 4, ctypes.byref(w), ctypes.byref(s)) == capi.EINVAL
    assert call(128, 100, 100, 0, 4, 3, 1, 256, items, 4, ctypes.byref(w), ctypes.byref(s)) == capi.EINVAL
    assert call(128, 8192, 8192, 0, 24, 6, 1, 256, items, 4, ctypes.byref(w), ctypes.byref(s)) == capi.ELIMIT


@pytest.mark.parametrize("head_dim", [64, 128, 256])
def test_the_prefill_workspace_has_room_for_parts_only_where_tiles_are_split(library, head_dim):
    """Angles and queries, and behind them the partial results of tiles whose keys are
    shared out: never for rows that are more than half of the keys a sequence can have,
    nor for more tiles than the lists hold."""
    def aligned(n):
        return -(-n // 256) * 256
    rotary, heads, kv_heads = 32, 24, 4
    def parts(length, capacity):
        p = capi.attention_params(heads, kv_heads, head_dim, rotary, capacity=capacity)
        base = 2 * aligned(length * rotary // 2 * 4) + aligned(length * heads * head_dim * 2)
        return library.pluto_hip_gqa_prefill_workspace_bytes(ctypes.byref(p), length) - base
    for length, capacity in [(8192, 8192), (1024, 1024), (1024, 2047), (513, 1025), (20, 1000), (20, 20),
                             (20000, 200000)]:
        assert parts(length, capacity) == 0, (length, capacity)
    for length, capacity in [(1024, 2048), (20, 1024), (1531, 3840)]:
        # at most 384 parts, each a tile's rows of outputs and two numbers a row
        rows = min(length, tile_rows(head_dim))
        want = 0 if head_dim == 64 else aligned(384 * rows * (head_dim + 2) * 4)
        assert parts(length, capacity) == want, (length, capacity)


PARTS = 384


def split(library, head_dim, q_rows, start, query_heads, group, resident=256):
    """(partitions, lists of (tile, begin, end, slot), tiles in parts) or None."""
    entries, first = (ctypes.c_uint16 * (4 * PARTS))(), (ctypes.c_uint16 * 257)()
    tiles = (ctypes.c_uint16 * (3 * PARTS // 2))()
    partitions, count = ctypes.c_int(-1), ctypes.c_int(-1)
    status = library.pluto_hip_test_forward_split(
        head_dim, q_rows, start + q_rows, start, query_heads, group, resident, entries, first, tiles,
        PARTS, ctypes.byref(partitions), ctypes.byref(count))
    assert status == 0
    if partitions.value == 0:
        return None
    lists = [[tuple(entries[4 * e:4 * e + 4]) for e in range(first[j], first[j + 1])]
             for j in range(256 // partitions.value)]
    return partitions.value, lists, [tuple(tiles[3 * i:3 * i + 3]) for i in range(count.value)]


def check_split(library, head_dim, q_rows, start, query_heads, group):
    made = split(library, head_dim, q_rows, start, query_heads, group)
    if made is None:
        return False
    partitions, lists, tiles = made
    kv_heads, q_tiles = query_heads // group, -(-q_rows // tile_rows(head_dim))
    assert partitions in (1, 2, 4, 8) and kv_heads % partitions == 0
    assert q_rows <= (start + q_rows) // 2
    items = q_tiles * query_heads // partitions
    entries = [e for part in lists for e in part]
    assert len(entries) <= PARTS

    def key_tiles(tile):
        last = min((tile % q_tiles + 1) * tile_rows(head_dim), q_rows) - 1
        return -(-(start + last + 1) // 64)

    # every key tile of every query tile once, whole tiles without a slot
    ranges = {}
    for tile, begin, end, slot in entries:
        assert tile < items and begin < end
        ranges.setdefault(tile, []).append((begin, end, slot))
    assert sorted(ranges) == list(range(items))
    parts = {tile: (slot, count) for tile, slot, count in tiles}
    assert len(parts) == len(tiles)
    used = []
    for tile, pieces in ranges.items():
        pieces.sort()
        assert pieces[0][0] == 0 and pieces[-1][1] == key_tiles(tile)
        assert all(a[1] == b[0] for a, b in zip(pieces, pieces[1:]))
        if pieces[0][2] == NO_ITEM:
            assert len(pieces) == 1 and tile not in parts
            continue
        # the parts' slots follow each other in the order of their keys
        assert [p[2] for p in pieces] == list(range(parts[tile][0], parts[tile][0] + parts[tile][1]))
        used += [p[2] for p in pieces]
        # all rows of the tile see all keys of every part but the last
        first_row = tile % q_tiles * tile_rows(head_dim)
        assert all(end * 64 <= start + first_row + 1 for _, end, _ in pieces[:-1])
    assert sorted(used) == list(range(len(used))) and 0 < len(used) * partitions <= PARTS
    assert len(parts) == sum(1 for pieces in ranges.values() if pieces[0][2] != NO_ITEM)
    # what the split is for: the fullest list carries less than it would with whole tiles
    def load(part):
        return sum(end - begin + 8 + (3 if slot != NO_ITEM else 0) for _, begin, end, slot in part)
    whole = [0] * len(lists)
    for tile in sorted(range(items), key=key_tiles, reverse=True):
        at = whole.index(min(whole))
        whole[at] += key_tiles(tile) + 8
    assert max(load(part) for part in lists) < max(whole)
    return True


def test_tiles_in_parts_cover_every_key_once(library):
    assert check_split(library, 256, 34, 7336, 24, 6)
    assert check_split(library, 256, 1531, 2309, 24, 6)
    rng = random.Random(11)
    made = 0
    for _ in range(600):
        group = rng.choice([1, 2, 3, 6, 8])
        kv_heads = rng.choice([1, 2, 4, 8, 16, 3, 5, 12])
        q_rows = rng.choice([rng.randint(1, 64), rng.randint(1, 600), rng.randint(1, 3000)])
        start = rng.choice([q_rows, rng.randint(0, 3000), rng.randint(3000, 60000)])
        made += bool(check_split(library, rng.choice([128, 256]), q_rows, start, group * kv_heads, group))
    assert made > 150    # the sample does split


def test_when_tiles_are_not_split(library):
    assert split(library, 256, 1024, 0, 24, 6) is None            # rows are all the keys
    assert split(library, 256, 1024, 1023, 24, 6) is None         # more than half of them
    assert split(library, 256, 34, 7336, 24, 6, resident=250) is None   # not the chip the lists are for
    assert split(library, 128, 20000, 200000, 24, 6) is None      # more tiles than the lists hold
    buffers = [(ctypes.c_uint16 * n)() for n in (4 * PARTS, 257, 3 * PARTS // 2)]
    a, b = ctypes.c_int(), ctypes.c_int()
    def call(head_dim, heads, group, capacity):
        return library.pluto_hip_test_forward_split(head_dim, 34, 7370, 7336, heads, group, 256, *buffers,
                                                    capacity, ctypes.byref(a), ctypes.byref(b))
    assert call(64, 24, 6, PARTS) == capi.EINVAL and call(256, 24, 5, PARTS) == capi.EINVAL
    assert call(256, 24, 6, PARTS - 1) == capi.ELIMIT
