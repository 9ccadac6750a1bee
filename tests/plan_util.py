"""attn_plan.hpp (the kernels' address rules and launch choices) built for the
host and loaded through ctypes."""
import ctypes
import functools
import os
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))


@functools.lru_cache(maxsize=None)
def load():
    with tempfile.TemporaryDirectory() as d:
        so = os.path.join(d, "plan.so")
        subprocess.run(["g++", "-O1", "-std=c++17", "-Wall", "-Werror", "-shared", "-fPIC", "-o", so,
                        os.path.join(HERE, "plan_shim.cpp")], check=True)
        lib = ctypes.CDLL(so)
    u32, i32, i64 = ctypes.c_uint32, ctypes.c_int32, ctypes.c_int64
    lib.tile_base.restype = u32
    lib.tile_base.argtypes = [i32, i32, u32]
    lib.range_shift.argtypes = [i32, i32]
    lib.burst_offset.restype = u32
    lib.burst_offset.argtypes = [u32, u32, u32, i32, i32]
    lib.prefill_split.argtypes = [i32] * 10 + [i64, i32]
    return lib


def prefill_split(hd, n_head, n_kv, T, kv_len, *, n_seq=1, keys=None, window=0, f32=False, row_stride=0, cus=256):
    """The split an 8-wave prompt launch takes (keys: a round's [begin, end))."""
    a, b = keys or (0, kv_len)
    return load().prefill_split(hd, n_head, n_kv, n_seq, T, kv_len, a, b, window, int(f32), row_stride, cus)
