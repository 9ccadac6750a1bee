"""Ring caches that have not wrapped: rows after a sequence's last key hold
whatever the allocation held (NaN here) and are no part of any result.
Against the CPU oracle, with the tolerances of its f32 and f16 outputs."""
import pytest
import torch

from pelica_amd import workloads as wl
from tests.gpu_util import as_f64, gpu_run, oracle_run
from tests.refimpl import assert_close

pytestmark = pytest.mark.gpu


def _ring(inp, L, cap, kv):
    r = torch.full((cap, *kv.shape[1:]), float("nan"), dtype=torch.float16, device="cuda")
    idx = torch.arange(max(0, L - cap), L, device="cuda")
    r[idx % cap] = kv[idx]
    return r


@pytest.mark.parametrize("kind,hd,n_head,n_kv,T,L,window,cap,f32", [
    ("decode", 64, 64, 8, 1, 40, 128, 200, False),
    ("decode", 64, 64, 8, 4, 130, 128, 131, False),     # one row never written
    ("decode", 128, 32, 4, 2, 100, 0, 300, False),
    ("decode", 64, 64, 8, 1, 1500, 2000, 2200, False),  # several splits
    ("decode", 64, 24, 8, 2, 30, 20, 40, False),        # a ring shorter than a block
    ("prefill", 64, 64, 8, 20, 40, 128, 200, False),    # one row tile a wave, resident tiles
    ("prefill", 64, 64, 8, 20, 40, 128, 200, True),
    ("prefill", 64, 64, 8, 2500, 2500, 128, 2700, False),  # the sliding-window kernel
    ("prefill", 64, 64, 8, 2500, 2500, 128, 2700, True),   # two row tiles a wave
    ("prefill", 64, 64, 8, 100, 100, 500, 700, False),  # one row tile a wave, streamed tiles
    ("prefill", 64, 64, 8, 100, 100, 500, 700, True),
    ("prefill", 128, 32, 4, 100, 100, 300, 500, False),
    ("prefill", 128, 32, 4, 100, 100, 0, 300, True),
    ("prefill", 64, 64, 8, 90, 210, 0, 230, False),
])
def test_rows_never_written(kind, hd, n_head, n_kv, T, L, window, cap, f32):
    cfg = wl.AttnConfig("ringnw", kind, n_head, n_kv, hd, L, q_tokens=T, window=window, sinks=hd == 64, seed=L + cap)
    inp = wl.make_inputs(cfg, "cuda")
    print(f"[case] rows never written {kind} hd{hd} h{n_head}/{n_kv} T{T} L{L} window{window} cap{cap} f32 {f32}",
          flush=True)
    ref = as_f64(oracle_run(inp))
    if f32:
        inp.q = inp.q.float()
    got = gpu_run(inp, ring_cap=cap, k=_ring(inp, L, cap, inp.k), v=_ring(inp, L, cap, inp.v))
    assert_close(as_f64(got), ref, what="ring rows")


@pytest.mark.parametrize("T,L,window,cap,f32", [
    (100, 2000, 500, 607, False),   # one row tile a wave over streamed tiles, a ring that has wrapped
    (300, 1500, 1000, 1300, True),
    (40, 900, 200, 256, False),     # tiles that wrap inside
    (1, 400, 700, 701, True),
])
def test_streamed_ring_tiles_of_one_row_tile(T, L, window, cap, f32):
    cfg = wl.AttnConfig("ringst", "prefill", 64, 8, 64, L, q_tokens=T, window=window, sinks=True, seed=T + cap)
    inp = wl.make_inputs(cfg, "cuda")
    print(f"[case] streamed ring tiles T{T} L{L} window{window} cap{cap} f32 {f32}", flush=True)
    ref = as_f64(oracle_run(inp))
    if f32:
        inp.q = inp.q.float()
    got = gpu_run(inp, ring_cap=cap, k=_ring(inp, L, cap, inp.k), v=_ring(inp, L, cap, inp.v))
    assert_close(as_f64(got), ref, what="streamed ring tiles")
