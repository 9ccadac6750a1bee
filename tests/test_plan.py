"""The kernels' address rules and launch choices (pelica_amd/csrc/attn_plan.hpp),
run on the host."""
import random

import pytest

from tests import plan_util


@pytest.fixture
def plan():
    return plan_util.load()


def _spans():
    """(rows, bytes per row) of accepted caches: rows + 128 rows below 4 GiB,
    the widest and the longest among them."""
    rng = random.Random(1)
    for stride in (128, 1024, 2048, 8192, 1 << 20, 4 << 20, 16 << 20, 32 << 20):
        most = ((1 << 32) - 1) // stride - 128
        for rows in {most, most - 1, most // 2, 1, *(rng.randint(1, max(1, most)) for _ in range(20))}:
            if rows >= 1 and (rows + 128) * stride < 1 << 32:
                yield rows, stride


def test_unwanted_tile_reads_nothing(plan):
    # every lane of a 64-row tile past the last one: at or past the end of the
    # rows (the buffer reads nothing there), with no wrap around 2^32
    n = 0
    for rows, stride in _spans():
        nrec = rows * stride
        base = plan.tile_base(0, rows + 64, stride)
        for key in (0, 1, 31, 63):
            for piece in (0, 16, min(stride, 256) - 16):  # (of a head's row)
                off = base + key * stride + piece
                assert nrec <= off < 1 << 32, (rows, stride, key)
                n += 1
    assert n > 1000


def test_wanted_tile_starts_at_its_row(plan):
    for rows, stride in _spans():
        for first in {0, rows // 2, rows - 1}:
            assert plan.tile_base(1, first, stride) == first * stride


def test_key_range_blocks_start_at_its_rows(plan):
    # every 64-key block of a range starts at one of its rows or past them, so
    # no row's offset, less the instruction's own part, falls below zero; and
    # the range lies in as few splits as its keys fill
    rng = random.Random(2)
    for _ in range(3000):
        split = 64 * rng.choice((1, 1, 2, 3, 4, 7, 16, 100))
        begin = rng.randrange(40000)
        keys = rng.randint(1, 9000)
        shift = plan.range_shift(begin, split)
        lo = begin + shift  # the position of row 0
        assert 0 <= shift < split
        first_split, last_split = lo // split, (lo + keys - 1) // split
        assert last_split - first_split + 1 == -(-keys // split)
        hd = rng.choice((64, 128))
        per_load, stride = 512 // hd, hd * 2 * rng.choice((1, 4, 8, 32, 4096))
        first = first_split * split - lo  # the first block's row
        b = first * stride % (1 << 32)
        j, e, lane = 4 * rng.randrange(hd // 32), rng.randrange(4), rng.randrange(64)
        lane_off = lane // (hd // 8) * stride + lane % (hd // 8) * 16
        row = first + per_load * (j + e) + lane // (hd // 8)
        assert row >= 0
        off = plan.burst_offset(lane_off, b, per_load * stride, j, e)
        assert off + 1024 * e == row * stride + lane % (hd // 8) * 16


# us of every split (1, 2, 4, ...), as measured on an MI355X
_MEASURED = [
    # windows of several thousand keys: a block walks its window, not the cache
    (dict(hd=128, n_head=40, n_kv=8, T=1024, kv_len=20688, window=1100), (37.1, 50.4, 49.4, 74.9)),
    (dict(hd=128, n_head=40, n_kv=8, T=1024, kv_len=18369, window=8000, f32=True), (197.9, 235.4, 225.0, 335.2)),
    (dict(hd=64, n_head=24, n_kv=8, T=1024, kv_len=24149, window=1500), (54.5, 34.2, 24.9, 41.4, 39.1)),
    # one chunk of keys: nothing to divide
    (dict(hd=64, n_head=64, n_kv=8, T=4, kv_len=21, f32=True), (7.2, 9.0, 10.2, 10.9, 8.7)),
    (dict(hd=64, n_head=24, n_kv=8, T=16, kv_len=16, f32=True), (7.5, 9.4, 10.7, 11.7, 8.5)),
    # ... but the queries to bring in
    (dict(hd=128, n_head=32, n_kv=2, T=16, kv_len=16, f32=True), (12.7, 12.3, 11.9, 9.3)),
    # kv heads that are no multiple of the XCDs: some get the long blocks
    (dict(hd=128, n_head=32, n_kv=2, T=558, kv_len=558, n_seq=2, f32=True), (26.7, 32.6, 40.1, 46.7)),
    (dict(hd=128, n_head=32, n_kv=4, T=1176, kv_len=1176), (36.6, 39.9, 39.7, 62.3)),
    # few rows over many keys
    (dict(hd=64, n_head=64, n_kv=8, T=512, kv_len=19817, f32=True), (496.7, 269.4, 190.9, 219.7, 276.9)),
    (dict(hd=128, n_head=32, n_kv=4, T=85, kv_len=10815, keys=(825, 10815), f32=True), (230.1, 124.3, 94.2, 75.5)),
    (dict(hd=128, n_head=32, n_kv=4, T=518, kv_len=6246, keys=(3439, 6246)), (77.8, 48.3, 59.0, 69.6)),
    (dict(hd=64, n_head=64, n_kv=8, T=25, kv_len=4270), (110.6, 61.9, 39.9, 26.1, 18.5)),
    # a full chip
    (dict(hd=64, n_head=64, n_kv=8, T=3196, kv_len=3196), (107.2, 121.3, 155.7, 218.3, 273.1)),
]


@pytest.mark.parametrize("call,times", _MEASURED)
def test_split_is_a_fast_one(call, times):
    split = plan_util.prefill_split(**call)
    assert times[split.bit_length() - 1] <= 1.1 * min(times), split


def test_split_counts_the_keys_a_window_shows():
    # keys before every window change nothing
    rng = random.Random(4)
    for _ in range(500):
        n_head, n_kv, hd = rng.choice([(64, 8, 64), (32, 4, 128), (40, 8, 128), (16, 16, 128), (24, 8, 64)])
        T, window, f32 = rng.randint(1, 3000), rng.randint(1025, 9000), rng.random() < 0.5
        near = plan_util.prefill_split(hd, n_head, n_kv, T, T + window, window=window, f32=f32)
        far = plan_util.prefill_split(hd, n_head, n_kv, T, T + window + rng.randint(1, 200000), window=window, f32=f32)
        assert near == far, (n_head, n_kv, hd, T, window)


def test_split_is_one_the_launch_has():
    rng = random.Random(5)
    for _ in range(3000):
        hd = rng.choice((64, 128))
        rows = 512 if hd == 64 else 256
        hpk = rng.choice((1, 2, 3, 5, 8, 16, 40, 100, rows))
        n_kv, n_seq, T = rng.randint(1, 40), rng.choice((1, 1, 2, 9, 64)), int(2 ** rng.uniform(0, 17))
        kv_len = T + rng.choice((0, rng.randint(0, 300000)))
        b = rng.randint(1, kv_len)
        keys = rng.choice((None, (rng.randrange(b), b)))
        split = plan_util.prefill_split(hd, hpk * n_kv, n_kv, T, kv_len, n_seq=n_seq, keys=keys,
                                        window=rng.choice((0, 0, 1025, 5000)), f32=rng.random() < 0.5,
                                        cus=rng.choice((256, 304, 38, 1)))
        assert split in ((1, 2, 4, 8, 16) if hd == 64 else (1, 2, 4, 8)) and rows // split >= hpk
