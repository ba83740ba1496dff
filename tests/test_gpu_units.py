"""The unit launch (units.hip) against the CPU oracle (attend, crates/engine/model/src/forward.rs:585-807)
and against the general path on the same call: runs of drafted tokens on every page type, prompts on
the head widths the prefill kernel has no instance for, and every row of the row layout and of f32
pages, at the sizes where its tiling can go wrong (one key, ends of 16-key tiles and 32-key steps,
column blocks that start inside a token, groups that do not divide 16, keys shared by one to eight
waves, units cut into key pieces, windows, larger blocks).

The general path (explicit split settings keep every call off the unit launch) carries Q and the
weights to the same 16 bits or more: Q's last kept bit is 2^-17 of it on bf16 pages, so scores of
|s| <= 8 differ by 2^-13 at most and typically by their root, outputs by less than 2e-4 of the row."""

import numpy as np
import pytest

from conftest import TOL, row_rel_err
from llmario_amd.kv import Layer
from llmario_amd.workloads import small
from test_gpu_parity import THREADS, pair, run_gpu

pytestmark = pytest.mark.gpu

CASES = [
    # drafted tokens (few columns per unit) on the matrix-core page types
    ("f16", (32, 8, 128, 128), [2000, 1994, 2041, 300], [6, 7, 5, 1], 0, 16),
    ("bf16", (40, 8, 128, 128), [3000, 1703, 905], [7, 6, 4], 0, 32),
    ("q8_0", (32, 8, 128, 128), [2500, 1994, 31], [6, 7, 5], 0, 16),
    ("f16", (32, 32, 64, 64), [1210, 15, 0], [7, 2, 1], 0, 64),
    ("bf16", (32, 32, 64, 64), [1210, 900], [7, 7], 500, 16),
    ("q8_0", (32, 32, 64, 64), [1215, 400], [7, 5], 0, 16),
    ("f16", (64, 8, 128, 128), [9000], [7], 0, 16),          # one long context: key pieces
    ("f16", (12, 2, 128, 128), [30000], [4], 0, 16),         # few KV heads: a unit in up to 64 pieces
    ("f16", (4, 1, 80, 80), [30000], [1], 0, 16),
    ("bf16", (32, 1, 80, 80), [20000, 50], [1, 2], 0, 16),   # groups wider than a unit, in pieces
    ("f16", (142, 2, 64, 64), [20000], [3], 0, 32),
    ("f32", (64, 2, 128, 128), [9000], [1], 0, 16),
    # prompts on widths without a prefill instance
    ("bf16", (16, 4, 256, 256), [1000, 0, 40], [150, 190, 1], 300, 16),
    ("f16", (64, 2, 256, 256), [60], [290], 0, 16),          # 32 query heads per KV head
    ("q8_0", (16, 4, 256, 256), [250, 9], [130, 131], 0, 32),
    ("q8_0", (8, 8, 192, 192), [100], [140], 0, 16),
    ("f16", (16, 8, 192, 192), [300], [123], 0, 16),
    ("bf16", (32, 8, 192, 128), [700], [61], 0, 16),
    ("f16", (12, 4, 96, 96), [0, 17], [333, 100], 0, 16),
    ("bf16", (8, 4, 32, 32), [64], [401], 129, 16),
    # the row layout
    ("f16", (32, 32, 80, 80), [299, 1, 0, 500], [120, 2, 1, 1], 0, 16),
    ("bf16", (8, 2, 80, 80), [1500, 16], [1, 35], 0, 16),
    ("f16", (12, 4, 112, 112), [777, 63], [3, 1], 400, 32),
    ("bf16", (8, 8, 40, 40), [95], [33], 0, 16),
    ("f16", (16, 4, 64, 128), [2000], [1], 0, 64),
    ("bf16", (4, 1, 200, 200), [700], [9], 0, 16),
    ("f16", (8, 2, 256, 128), [31, 32], [1, 1], 0, 16),
    ("f16", (4, 4, 8, 8), [37], [20], 0, 16),
    # row-layout widths inside an instance's
    ("f16", (4, 2, 160, 160), [300, 9], [45, 1], 0, 16),
    ("bf16", (4, 2, 160, 144), [300, 9], [45, 1], 0, 32),
    ("bf16", (16, 4, 104, 104), [500], [40], 0, 16),
    ("bf16", (4, 1, 120, 128), [1900, 30], [1, 3], 200, 16),
    ("f16", (8, 2, 256, 200), [90], [30], 0, 16),
    # more units than the device holds waves: several rounds, the longest first
    ("bf16", (16, 4, 256, 256), [0, 300], [1500, 900], 200, 16),
    ("f32", (8, 8, 64, 64), [0, 30], [4200, 4100], 64, 16),
    # f32 pages
    ("f32", (8, 8, 64, 64), [0, 255], [70, 1], 0, 16),
    ("f32", (16, 2, 128, 128), [600, 900, 15], [1, 1, 1], 0, 16),
    ("f32", (16, 1, 256, 256), [300, 90], [17, 40], 100, 32),
    ("f32", (12, 4, 96, 96), [3000], [1], 0, 16),            # key pieces
    ("f32", (4, 2, 100, 36), [50], [31], 0, 16),
]


# every instance the library compiles: (page type, hd, hdv, 16-column blocks)
TILES = [(d, d) for d in (32, 64, 96, 128, 192, 256)] + [(192, 128)]
INSTANCES = [(kv, hd, hdv, nb) for kv in ("f16", "bf16") for hd, hdv in TILES for nb in (1, 2)]
INSTANCES += [("q8_0", d, d, nb) for d, nb in ((64, 1), (64, 2), (128, 1), (128, 2), (192, 1), (256, 1))]
INSTANCES += [(kv, d, d, nb) for kv in ("f16", "bf16") for d, nb in ((56, 1), (56, 2), (88, 1), (88, 2), (120, 1), (184, 1), (248, 1))]
INSTANCES += [("f32", d, d, nb) for d, nb in ((64, 1), (64, 2), (128, 1), (128, 2), (256, 1))]


def launches(hc, f):
    hc.kernel_times()
    hc.set_timing(True)
    r = f()
    kt = hc.kernel_times()
    hc.set_timing(False)
    return r, kt


@pytest.mark.parametrize("kv,geo,prior,new,window,bt", CASES,
                         ids=[f"{c[0]}-{'x'.join(map(str, c[1]))}-{'_'.join(map(str, c[3]))}" for c in CASES])
def test_units_match_the_oracle_and_the_general_path(cuda, kv, geo, prior, new, window, bt):
    w = small("un", kv, Layer(*geo), prior=prior, new=new, window=window, seed=81, block_tokens=bt)
    hc, oc, q = pair(w)
    q = np.random.default_rng(83).standard_normal(q.shape).astype(np.float32)   # all f32 bits
    got, kt = launches(hc, lambda: run_gpu(hc, w, q))
    assert kt["prefill"][1] == 1 and kt["decode"][1] == 0 and kt["mixed"][1] == 0, kt
    assert np.isfinite(got).all()
    ref = oc.attend(0, w.segments(), q, w.scale, w.window, THREADS)
    err = row_rel_err(got, ref)
    hc.set_tuning(prefill_min_rows=1 << 32, decode_min_tiles=8)
    gen, kt = launches(hc, lambda: run_gpu(hc, w, q))
    assert kt["prefill"][1] == 0 and kt["decode"][1] == 1, kt
    diff = row_rel_err(got, gen)
    print(f"{kv} {geo}: oracle {err:.3e}, general path {diff:.3e}")
    assert err <= TOL[kv] and diff <= (2e-5 if kv == "f32" else 2e-4), (err, diff)


@pytest.mark.parametrize("kv,geo", [("f16", (8, 2, 80, 80)), ("bf16", (8, 2, 80, 80)), ("f32", (8, 4, 64, 64))])
def test_units_take_any_scale_of_q(cuda, kv, geo):
    """Row-layout and f32 pages never had a range limit on Q: 2^30 larger and smaller than usual with
    the scale the other way round, the scores and so the outputs are the same."""
    w = small("us", kv, Layer(*geo), prior=[200], new=[9], seed=85)
    hc, oc, q = pair(w)
    q = np.random.default_rng(87).standard_normal(q.shape).astype(np.float32)
    base = run_gpu(hc, w, q)
    scale = w.scale
    for e in (30, -30):
        w.scale = scale * 2.0 ** -e
        got = run_gpu(hc, w, (q * np.float32(2.0 ** e)).astype(np.float32))
        err = row_rel_err(got, base)
        print(f"{kv} q x 2^{e}: {err:.3e}")
        assert err <= 1e-6, err   # powers of two: the same roundings


@pytest.mark.parametrize("kv,geo", [("f16", (8, 2, 80, 80)), ("bf16", (4, 4, 40, 40)), ("f32", (8, 4, 64, 64))])
@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_a_row_ignores_values_it_does_not_see(cuda, kv, geo, bad):
    """V of one position is not finite: the rows before it (same tile, same unit) and, beyond the
    window, the rows after it are as they are without it; the rows that see it are not finite."""
    import torch

    at, window = 70, 40
    w = small("uv", kv, Layer(*geo), prior=[50], new=[70], window=window, seed=89)
    hc, oc, q = pair(w)
    base = run_gpu(hc, w, q)
    L = w.layer
    k, v = (torch.empty((1, L.n_kv * d), device="cuda") for d in (L.hd, L.hdv))
    hc.gather(0, [(0, 0, 1, at)], k, v)
    v[:] = bad
    hc.store(0, [(0, 0, 1, at)], k, v)
    got = run_gpu(hc, w, q)
    pos = 50 + np.arange(70)
    sees = (pos >= at) & (pos < at + window)
    assert np.array_equal(got[~sees], base[~sees])
    assert not np.isfinite(got[sees]).any()


# f16 / bf16 tiles: runs of drafted tokens across a tile's end, prompts at either edge of a window.
# 1e5 is beyond f16, in which the tiles' products are taken.
@pytest.mark.parametrize("kv,geo,prior,new,window,at", [
    ("f16", (32, 8, 128, 128), 3005, 7, 0, 3009), ("bf16", (32, 8, 128, 128), 3005, 7, 0, 3009),
    ("f16", (32, 32, 64, 64), 3005, 6, 0, 3010), ("bf16", (16, 4, 256, 256), 1000, 70, 1000, 1040),
    ("f16", (16, 4, 256, 256), 1000, 70, 1000, 30), ("bf16", (12, 4, 96, 96), 1000, 90, 0, 1017)])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), float("nan"), 1e5])
def test_a_row_on_tiles_ignores_values_it_does_not_see(cuda, kv, geo, prior, new, window, at, bad):
    import torch

    w = small("ut", kv, Layer(*geo), prior=[prior] * 4, new=[new] * 4, window=window, seed=91)
    hc, oc, q = pair(w)
    base, kt = launches(hc, lambda: run_gpu(hc, w, q))
    assert kt["prefill"][1] == 1 and kt["decode"][1] == 0, kt
    L = w.layer
    k, v = (torch.empty((1, L.n_kv * d), device="cuda") for d in (L.hd, L.hdv))
    hc.gather(0, [(1, 0, 1, at)], k, v)
    v[:] = bad
    hc.store(0, [(1, 0, 1, at)], k, v)
    got = run_gpu(hc, w, q)
    pos = prior + np.arange(4 * new) - new
    sees = (np.arange(4 * new) // new == 1) & (pos >= at)
    if window:
        sees &= pos < at + window
    assert 0 < sees.sum() < new
    assert np.array_equal(got[~sees], base[~sees])
    assert not np.isfinite(got[sees]).any()


@pytest.mark.parametrize("kv,geo,prior,new", [
    ("f16", (32, 8, 128, 128), [16000], [4]), ("q8_0", (32, 8, 128, 128), [16000], [4]), ("bf16", (16, 4, 256, 256), [9000], [5]),
    ("f16", (8, 2, 80, 80), [16000], [1]), ("f32", (64, 2, 128, 128), [9000], [1]),
    ("f16", (32, 8, 128, 128), [2000, 1500, 1700, 1900], [6, 7, 5, 6])])
def test_allocation_free_calls(cuda, kv, geo, prior, new):
    """lmh_attend_noalloc through the unit launch, in pieces (one long context) and whole."""
    import torch

    w = small("ua", kv, Layer(*geo), prior=prior, new=new, seed=105)
    hc, oc, q = pair(w)
    ref = oc.attend(0, w.segments(), q, w.scale, w.window, THREADS)
    qd, out = torch.from_numpy(q).cuda(), torch.full((q.shape[0], geo[0], geo[3]), float("nan"), device="cuda")
    hc.attend_noalloc(0, w.segments(), qd, out, w.scale, w.window)
    torch.cuda.synchronize()
    err, diff = row_rel_err(out.cpu().numpy(), ref), row_rel_err(out.cpu().numpy(), run_gpu(hc, w, q))
    print(f"{kv} {geo}: oracle {err:.3e}, attend {diff:.3e}")
    assert err <= TOL[kv] and diff <= (1e-5 if kv == "f32" else 2e-4), (err, diff)


def test_first_calls_of_a_cache_allocate_nothing(cuda):
    """The partials of a unit plan in pieces are reserved at creation: device memory stays as it was over
    a new cache's first calls, a longer one after a shorter one among them."""
    import gc
    import torch

    free = []
    for again in (False, True):   # the first cache's calls load the kernels
        w = small("uf", "f16", Layer(32, 8, 128, 128), prior=[1900 + 3 * i for i in range(24)], new=[4] * 24, seed=107)
        hc, oc, q = pair(w)
        qd = torch.from_numpy(q).cuda()
        out = torch.empty(q.shape[0], 32, 128, device="cuda")
        gc.collect()
        torch.cuda.synchronize()
        free = [torch.cuda.mem_get_info()[0]]
        for n in (8, 24):
            hc.attend(0, w.segments()[:n], qd[:4 * n], out[:4 * n], w.scale)
            torch.cuda.synchronize()
            free.append(torch.cuda.mem_get_info()[0])
    print(free)
    assert free[0] == free[1] == free[2]


@pytest.mark.parametrize("kv,hd,hdv,nb", INSTANCES, ids=[f"{i[0]}-{i[1]}x{i[2]}-{16 * i[3]}cols" for i in INSTANCES])
def test_every_instance(cuda, kv, hd, hdv, nb):
    """Runs of 7 rows on 14 or 28 columns of 8 KV heads (tile widths: long enough to be taken)."""
    from test_plan import contiguous_table
    from test_plan_units import wave_plan

    tiles = kv == "q8_0" or (kv != "f32" and (hd, hdv) in TILES)
    prior, geo = 5000 if tiles else 700, (16 * nb, 8, hd, hdv)
    w = small("ue", kv, Layer(*geo), prior=[prior, 33], new=[7, 7], seed=109)
    waves, merges, c = wave_plan(kv, *geo, 16, contiguous_table([prior + 7, 40], 16), w.segments(), 0, 256, 8, False)
    assert len(waves) and c.col_blocks == nb
    hc, oc, q = pair(w)
    q = np.random.default_rng(110).standard_normal(q.shape).astype(np.float32)
    got, kt = launches(hc, lambda: run_gpu(hc, w, q))
    assert kt["prefill"][1] == 1 and kt["decode"][1] == 0 and kt["mixed"][1] == 0, kt
    err = row_rel_err(got, oc.attend(0, w.segments(), q, w.scale, w.window, THREADS))
    print(f"{kv} {geo}: {err:.3e}")
    assert err <= TOL[kv], err
