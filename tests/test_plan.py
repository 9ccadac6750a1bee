"""The kernels' address rules (pelica_amd/csrc/attn_plan.hpp), run on the host."""
import ctypes
import os
import random
import subprocess

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="session")
def plan(tmp_path_factory):
    so = str(tmp_path_factory.mktemp("plan") / "plan.so")
    subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                    os.path.join(HERE, "plan_shim.cpp")], check=True)
    lib = ctypes.CDLL(so)
    u32, i32 = ctypes.c_uint32, ctypes.c_int32
    lib.tile_base.restype = u32
    lib.tile_base.argtypes = [i32, i32, u32]
    lib.range_shift.argtypes = [i32, i32]
    lib.burst_offset.restype = u32
    lib.burst_offset.argtypes = [u32, u32, u32, i32, i32]
    return lib


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
