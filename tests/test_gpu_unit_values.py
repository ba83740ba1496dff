"""The unit launch on values at the ends of the types' ranges, as each row has them when it walks its
own keys (attend, crates/engine/model/src/forward.rs:585-807)."""

import numpy as np
import pytest

from conftest import TOL, row_rel_err
from llmario_amd.kv import Layer
from llmario_amd.workloads import small
from test_gpu_cancelling import build
from test_gpu_parity import THREADS, pair, run_gpu
from test_gpu_q8_range import PROFILES
from test_gpu_units import launches

pytestmark = pytest.mark.gpu


def rewrite(hc, L, seq, at, n=1, k=None, v=None):
    """K and V of positions at .. at + n - 1 as the functions make them from what is there."""
    import torch

    kt, vt = (torch.empty((n, L.n_kv * d), device="cuda") for d in (L.hd, L.hdv))
    hc.gather(0, [(seq, 0, n, at)], kt, vt)
    if k:
        k(kt)
    if v:
        v(vt)
    hc.store(0, [(seq, 0, n, at)], kt, vt)


def unit_run(hc, w, q):
    got, kt = launches(hc, lambda: run_gpu(hc, w, q))
    assert kt["prefill"][1] == 1 and kt["decode"][1] == 0 and kt["mixed"][1] == 0, kt
    return got


# q8_0 tiles: runs of drafted tokens across a tile's end, prompts at either edge of a window. 1e7 is
# beyond an f16 scale (8.3e6); 1e6 is held, with a scale 5e5 times the other keys'.
@pytest.mark.parametrize("geo,prior,new,window,at", [
    ((32, 8, 128, 128), 3005, 7, 0, 3009), ((32, 32, 64, 64), 3005, 6, 0, 3010),
    ((16, 4, 256, 256), 1000, 70, 1000, 1040), ((16, 4, 256, 256), 1000, 70, 1000, 30),
    ((8, 8, 192, 192), 5, 90, 0, 20)])
@pytest.mark.parametrize("bad", [float("inf"), float("-inf"), 1e7, 1e6])
def test_a_row_on_q8_0_tiles_ignores_values_it_does_not_see(cuda, geo, prior, new, window, at, bad):
    w = small("uq", "q8_0", Layer(*geo), prior=[prior] * 4, new=[new] * 4, window=window, seed=93)
    hc, oc, q = pair(w)
    base = unit_run(hc, w, q)
    rewrite(hc, w.layer, 1, at, v=lambda v: v.fill_(bad))
    got = unit_run(hc, w, q)
    pos = prior + np.arange(4 * new) - new
    sees = (np.arange(4 * new) // new == 1) & (pos >= at)
    if window:
        sees &= pos < at + window
    assert 0 < sees.sum() < new
    if bad == 1e6:   # the rows that see it make their unit run again: its other columns round anew
        assert np.isfinite(got).all()
        assert row_rel_err(got[~sees], base[~sees]) <= 1e-6
    else:
        assert np.array_equal(got[~sees], base[~sees])
        assert not np.isfinite(got[sees]).any()


@pytest.mark.parametrize("kv", ["f16", "bf16"])
def test_q_keeps_its_small_elements(cuda, kv):
    """One dim of Q is 2^14 times the others where K is zero: the outputs are those of a Q without it,
    to the rounding of the scores (|s| <= 16, sums of 80 products in f32: 2^-24 x 16 x 80^0.5 < 1e-5)."""
    w = small("up", kv, Layer(8, 2, 80, 80), prior=[400], new=[5], seed=103)
    hc, oc, q = pair(w)
    L = w.layer
    rewrite(hc, L, 0, 0, n=405, k=lambda k: k.view(-1, L.n_kv, L.hd)[:, :, 7].fill_(0.0))
    q = np.random.default_rng(104).standard_normal(q.shape).astype(np.float32)
    q[:, :, 7] = 0
    base = unit_run(hc, w, q)
    q[:, :, 7] = 2.0 ** 14
    got = unit_run(hc, w, q)
    assert row_rel_err(got, base) <= 1e-5


@pytest.mark.parametrize("kv,geo", [("f16", (8, 2, 80, 80)), ("bf16", (4, 4, 40, 40)), ("f16", (4, 1, 200, 200)),
                                    ("f32", (8, 4, 64, 64))])
def test_an_infinite_value_gives_an_infinite_output(cuda, kv, geo):
    """V of one position is +inf in some dims, -inf in others: every row that sees it, near (a masked
    step) or far, has exactly those in these dims, and its other dims untouched."""
    w = small("ui", kv, Layer(*geo), prior=[0], new=[300], seed=95)
    hc, oc, q = pair(w)
    base = unit_run(hc, w, q)
    L, at = w.layer, 70
    plus, minus = [d % L.hdv for d in (1, 8, 17, 33)], [d % L.hdv for d in (0, 15, 34)]

    def put(v):
        v.view(L.n_kv, L.hdv)[:, plus] = float("inf")
        v.view(L.n_kv, L.hdv)[:, minus] = float("-inf")

    rewrite(hc, L, 0, at, v=put)
    got = unit_run(hc, w, q)
    assert np.array_equal(got[:at], base[:at])
    seen, rest = got[at:], [d for d in range(L.hdv) if d not in plus + minus]
    assert (seen[:, :, plus] == np.inf).all() and (seen[:, :, minus] == -np.inf).all()
    assert np.array_equal(seen[:, :, rest], base[at:][:, :, rest])


@pytest.mark.parametrize("kv,geo", [("f16", (8, 2, 80, 80)), ("bf16", (8, 2, 80, 80)), ("f32", (8, 4, 64, 64))])
def test_a_score_of_minus_infinity_takes_no_weight(cuda, kv, geo):
    """K of one position is -inf in a dim where every q is positive: the outputs are finite, as the
    general path's."""
    w = small("uk", kv, Layer(*geo), prior=[100], new=[60], seed=97)
    hc, oc, q = pair(w)
    q = np.random.default_rng(98).standard_normal(q.shape).astype(np.float32)
    q[:, :, 3] = np.abs(q[:, :, 3]) + 0.01
    L = w.layer
    rewrite(hc, L, 0, 40, k=lambda k: k.view(L.n_kv, L.hd)[:, 3].fill_(float("-inf")))
    got = unit_run(hc, w, q)
    hc.set_tuning(prefill_min_rows=1 << 32, decode_min_tiles=8)
    gen = run_gpu(hc, w, q)
    assert np.isfinite(gen).all() and np.isfinite(got).all()
    assert row_rel_err(got, gen) <= (2e-5 if kv == "f32" else 2e-4)


@pytest.mark.parametrize("kv,geo", [("bf16", (8, 2, 80, 80)), ("f32", (8, 4, 64, 64))])
def test_values_near_the_types_largest(cuda, kv, geo):
    """V of about 1e36 (the largest is 3.4e38): no weighted value leaves the range of f32."""
    w = small("ul", kv, Layer(*geo), prior=[200], new=[9], seed=101)
    hc, oc, q = pair(w)
    rewrite(hc, w.layer, 0, 0, n=209, v=lambda v: v.mul_(1e36))
    got = unit_run(hc, w, q)
    hc.set_tuning(prefill_min_rows=1 << 32, decode_min_tiles=8)
    gen = run_gpu(hc, w, q)
    assert np.isfinite(gen).all() and np.isfinite(got).all()
    assert row_rel_err(got, gen) <= (2e-5 if kv == "f32" else 2e-4)


@pytest.mark.parametrize("geo,prior,new", [
    ((32, 8, 128, 128), [3000, 1500, 2700, 1900], [6, 7, 5, 6]), ((16, 8, 128, 128), [2900, 2500, 1400, 700], [7, 6, 7, 7]),
    ((32, 32, 64, 64), [3000, 1200], [6, 7]), ((8, 8, 192, 192), [100, 1400], [140, 33]), ((16, 4, 256, 256), [0, 1000], [131, 90])])
@pytest.mark.parametrize("profile", list(PROFILES))
def test_q8_0_scales_over_their_range(cuda, geo, prior, new, profile):
    """V blocks whose scales span f16's range, rising or falling along the sequence: a step's products can
    overflow what the first set, and the unit runs again (test_gpu_q8_range, for the decode items)."""
    import torch

    layer = Layer(*geo)
    hc, oc, segs, n_rows, rng = build("q8_0", layer, prior, new, 61, v_scale=PROFILES[profile])
    q = rng.standard_normal((n_rows, layer.n_head, layer.hd)).astype(np.float32)
    out = torch.full((n_rows, layer.n_head, layer.hdv), float("nan"), device="cuda")
    _, kt = launches(hc, lambda: hc.attend(0, segs, torch.from_numpy(q).cuda(), out, layer.hd ** -0.5))
    assert kt["prefill"][1] == 1 and kt["decode"][1] == 0 and kt["mixed"][1] == 0, kt
    got, ref = out.cpu().numpy(), oc.attend(0, segs, q, layer.hd ** -0.5, 0, THREADS)
    err = row_rel_err(got, ref)
    print(f"{geo} {profile}: {err:.3e}")
    assert bool(np.isfinite(got).all()) and err <= TOL["q8_0"], err
