"""tb_build_prefill_columns_work (host code, no GPU): every (query row, head, position) a
sequence's rows may see is covered by exactly one entry; padding entries have no rows; the
partition rule keeps rows whole when the step fills the GPU and never asks for more
scratch than the tiles did, past the static scratch."""
import os
import subprocess
import sys
import time

import numpy as np
import pytest

from tinybatch_amd.kv_cache import PagedKVCache
from tinybatch_amd.metadata import (TILE_PARTITION, ColumnsRoute, PrefillRoute, build_columns_work,
                                    build_step_metadata, columns_partition, columns_pay)


def covered(first, pos0, rows, hq, hkv, work, part):
    """How often each (row, head) meets each partition it has positions in."""
    rep = hq // hkv
    seen = [np.zeros((n, hq, -(-(p + n) // part)), dtype=int) for p, n in zip(pos0, rows)]
    for r0, seq, p0, n, col0, kvh, p, pc in work.tolist():
        if n == 0:
            continue
        assert (r0, p0, n, pc) == (first[seq], pos0[seq], rows[seq], part // 64)
        for col in range(col0, min(col0 + 128, n * rep)):
            seen[seq][col // rep, kvh * rep + col % rep, p] += 1
    for s, p0, n in zip(seen, pos0, rows):
        for r in range(n):
            mine = -(-(p0 + r + 1) // part)
            assert (s[r, :, :mine] == 1).all() and (s[r, :, mine:] <= 1).all()


@pytest.mark.parametrize("hq,hkv", [(14, 2), (32, 8), (5, 1), (4, 4)])
@pytest.mark.parametrize("xcds", [1, 8])
@pytest.mark.parametrize("part", [64, 512, 1 << 20])
def test_every_row_head_and_partition_once(hq, hkv, xcds, part):
    rows, pos0 = [16, 19, 64, 129, 300], [0, 45, 1000, 63, 2]
    first = np.concatenate([[0], np.cumsum(rows)[:-1]]).tolist()
    work = build_columns_work(first, range(5), pos0, rows, part, ColumnsRoute(hq, hkv, 64, xcds, 256))
    assert len(work) % xcds == 0
    covered(first, pos0, rows, hq, hkv, work, part)


def test_partitions():
    r = ColumnsRoute(14, 2, 64, 8, 256)
    assert columns_partition([0] * 4, [3251, 1746, 3738, 2168], r) > 3738         # enough rows: none split
    assert columns_partition([0], [600], r) >= 600                              # a merge would cost more than it saves
    p = columns_partition([3000] * 4, [20] * 4, r)
    assert p % 64 == 0 and p < TILE_PARTITION
    # a call without a workspace: shorter than the tiles' partition only within the static scratch
    slot = 14 * 66 * 4
    for pos0, n, other in ((9000, 1500, 0), (1000, 100, 0), (1000, 100, (32 << 20) // slot)):
        p = columns_partition([pos0], [n], r, other)
        slots = other + sum(-(-(pos0 + i + 1) // p) for i in range(n))
        assert p >= TILE_PARTITION or slots * slot <= 32 << 20
    with pytest.raises(RuntimeError):
        columns_partition([0], [0], r)


def test_metadata_counts_partitions_of_the_columns():
    r = ColumnsRoute(14, 2, 64, 8, 256)
    m = build_step_metadata(list(range(2000, 2040)) + [99], [(0, 40), (40, 41)], [list(range(128)), [200] * 7],
                            [2040, 100], block_size=16, num_blocks=256, partition_tokens=256, rows_per_item=2,
                            tile_prefill=True, columns_route=r)
    part = columns_partition([2000], [40], r)
    assert m.num_columns_work and m.num_prefill_tiles == 0 and m.num_work_items == 1
    assert np.diff(m.row_part_off_np).tolist() == [-(-(2001 + i) // part) for i in range(40)] + [1]
    assert m.split_rows_np[:, 0].tolist() == list(range(40))


def both_routes():
    """A 100-row prompt for tb_paged_prefill beside a 1000-row one for the column tiles."""
    return build_step_metadata(list(range(100)) + list(range(1000)), [(0, 100), (100, 1100)],
                               [list(range(7)), list(range(7, 70))], [100, 1000], block_size=16, num_blocks=70,
                               partition_tokens=256, rows_per_item=2, tile_prefill=True,
                               prefill_route=PrefillRoute(2, 64, 560, 8), columns_route=ColumnsRoute(14, 2, 64, 8, 256))


def test_column_rows_are_not_appended_by_the_attention():
    m = both_routes()
    assert m.num_prefill_work and m.num_columns_work and not m.num_work_items and not m.num_prefill_tiles
    assert not PagedKVCache._fusable(m) and not m.whole_prefills_only()
    only = build_step_metadata(list(range(100)), [(0, 100)], [list(range(7))], [100], block_size=16, num_blocks=7,
                               partition_tokens=256, prefill_route=PrefillRoute(2, 64, 560, 8))
    assert only.whole_prefills_only() and PagedKVCache._fusable(only)


@pytest.mark.parametrize("hq,hkv", [(14, 2), (28, 2), (7, 1), (4, 4), (32, 8)])
def test_other_heads_get_a_list_of_their_own(hq, hkv):
    """Metadata built for 14 / 2 heads, used with others: every (row, head) of the call once."""
    m = build_step_metadata(list(range(900, 1000)), [(0, 100)], [list(range(63))], [1000], block_size=16, num_blocks=63,
                            partition_tokens=256, columns_route=ColumnsRoute(14, 2, 64, 8, 256))
    work = m.columns_list(hq, hkv)
    assert (work is m.columns_work_np) == ((hq, hkv) == (14, 2))
    covered([0], [900], [100], hq, hkv, work, m.columns_partition)


def test_partition_of_very_long_prompts():
    """Contexts past 2^24 positions are taken; the rule's time grows with the tiles and not
    with their square (2^23 rows took 1.2 s when every length walked every tile; 1 ms now)."""
    r = ColumnsRoute(4, 4, 64, 8, 256)
    assert columns_partition([1 << 25], [32], r) > 0
    assert len(build_columns_work([0], [0], [1 << 25], [32], 1 << 26, r)) == 8
    t = time.perf_counter()
    assert columns_partition([0], [1 << 23], r) % 64 == 0
    assert time.perf_counter() - t < 0.3


@pytest.mark.parametrize("hq,hkv,d,dtype,prompts,others,want", [
    (14, 2, 64, 2, [(0, 40)], 4, False),              # tiles beside decode rows: one launch
    (14, 2, 64, 2, [(0, 700)], 4, False),
    (14, 2, 64, 2, [(0, 1500)] * 4, 4, True),
    (14, 2, 64, 2, [(8000, 300)], 4, True),           # as work items otherwise
    (14, 2, 64, 2, [(0, 700)] * 4, 0, False),
    (14, 2, 64, 2, [(0, 700)] * 16, 0, True),
    (14, 2, 64, 1, [(3000, 100)] * 12, 0, True),
    (8, 8, 64, 2, [(0, 850)] * 16, 0, False),         # one head per kv head
    (32, 8, 128, 2, [(0, 280)], 0, True),
    (32, 8, 128, 2, [(0, 40)], 4, False),
    (14, 2, 64, 0, [(0, 16)], 0, False),
    (14, 2, 64, 0, [(0, 100)] * 16, 0, True),
    (14, 2, 64, 0, [(1008, 16)], 8, False),
    (32, 8, 128, 0, [(0, 400)], 0, True),
    (14, 2, 64, 2, [], 4, False),
    (14, 2, 64, 2, [((1 << 30) - 10, 16)], 0, False)])   # past the work list's positions
def test_where_the_column_tiles_pay(hq, hkv, d, dtype, prompts, others, want):
    """Either side of the rule's lines, as both routes measured."""
    seqs = [(c, n) for c, n in prompts] + [(500, 1)] * others
    ends = np.cumsum([n for _, n in seqs]).tolist()
    slices = list(zip([0] + ends[:-1], ends))
    assert columns_pay(slices, [c + n for c, n in seqs], ColumnsRoute(hq, hkv, d, 8, 256, dtype), dtype != 0) == want


def test_rule_refuses_what_the_work_list_refuses():
    with pytest.raises(RuntimeError):
        columns_pay([(0, 16)], [100], ColumnsRoute(14, 4, 64, 8, 256), True)
    with pytest.raises(RuntimeError):
        columns_pay([(0, 16)], [100], ColumnsRoute(14, 2, 96, 8, 256), True)


def test_a_list_past_the_memory_is_an_error():
    """An allocation that fails behind the C entry is a status, not an exception out of it."""
    code = """
import ctypes, resource, sys
lib = ctypes.CDLL(sys.argv[1])
page = resource.getpagesize() * int(open("/proc/self/statm").read().split()[0])
resource.setrlimit(resource.RLIMIT_AS, (page + (256 << 20),) * 2)
one = lambda x: ctypes.byref(ctypes.c_int32(x))
n = ctypes.c_int32()
st = lib.tb_build_prefill_columns_work(one(0), one(0), one((1 << 30) - (1 << 20)), one(1 << 20), 1, 1, 1, 64, 8, 256,
                                       None, 0, ctypes.byref(n))
print("status", st)
"""
    from tinybatch_amd.build import LIB_PATH
    r = subprocess.run([sys.executable, "-c", code, LIB_PATH], capture_output=True, text=True, timeout=120,
                       env={**os.environ, "HIP_VISIBLE_DEVICES": ""})
    assert r.returncode == 0 and r.stdout.startswith("status -"), (r.returncode, r.stdout, r.stderr[-300:])
