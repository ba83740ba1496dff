"""Which calls lmh_attend's planner gives to the unit launch (units.hip) and which to the prefill and
decode kernels, on the CPU, over the forms the rule tells apart: page type and width (an instance or
none), layout, segment lengths, head group, block size, split settings. Every plan is also checked to
cover each row's keys once (check_plan: attend's ranges, crates/engine/model/src/forward.rs:585-807);
the GPU tests compare the two routes' outputs."""

import ctypes as C
from types import SimpleNamespace

import numpy as np
import pytest

from llmario_amd import _native as N
from test_plan import KV, NO_SLOT, check_plan, contiguous_table, plan

# kv, (n_head, n_kv, hd, hdv), block, prior, new, options, expected: "units", "items" (decode items
# alone) or "prefill" (prefill units, beside decode items if the call has decode rows)
FORMS = [
    ("f16", (32, 8, 128, 128), 16, [2000] * 4, [6] * 4, {}, "units"),
    ("f16", (32, 8, 128, 128), 16, [2000] * 4, [1] * 4, {}, "items"),        # decode rows alone
    ("f16", (32, 8, 128, 128), 16, [100] * 4, [2] * 4, {}, "items"),         # too little to share
    ("f16", (32, 8, 128, 128), 16, [2000] * 4, [6, 6, 6, 8], {}, "prefill"),   # one long segment
    ("f16", (32, 8, 128, 128), 16, [2000] * 4, [6] * 4, {"prefill_min_rows": 8}, "items"),
    ("f16", (32, 8, 128, 128), 16, [2000] * 4, [6] * 4, {"decode_min_tiles": 8}, "items"),
    ("q8_0", (32, 8, 128, 128), 32, [2000] * 4, [6] * 4, {}, "units"),
    ("bf16", (16, 4, 256, 256), 16, [500, 40], [200, 1], {}, "units"),       # no prefill instance
    ("f16", (12, 4, 96, 96), 64, [0], [500], {}, "units"),
    ("q8_0", (12, 4, 96, 96), 16, [100], [50], {}, "items"),                 # row layout, q8_0: no instance
    ("f16", (32, 32, 80, 80), 16, [700], [1], {}, "units"),                  # row layout, decode rows too
    ("bf16", (8, 2, 80, 80), 16, [15], [3], {}, "units"),
    ("f16", (8, 2, 100, 100), 16, [300], [5], {}, "items"),                  # width not a multiple of 8
    ("f16", (8, 2, 80, 80), 8, [300], [5], {}, "items"),                     # blocks under 16 positions
    ("f16", (8, 1, 512, 512), 16, [300], [5], {}, "items"),                  # wider than any instance
    ("f16", (16, 4, 64, 128), 16, [300], [1], {}, "units"),
    ("f32", (8, 8, 64, 64), 16, [255], [1], {}, "items"),
    ("f32", (8, 8, 64, 64), 16, [255], [2], {}, "units"),
    ("f32", (64, 8, 128, 128), 16, [900], [1], {}, "units"),                 # wide group, long row
    ("f32", (64, 8, 128, 128), 16, [200], [1], {}, "items"),
    ("f32", (8, 2, 100, 100), 16, [300], [1], {}, "units"),
    ("f32", (8, 2, 50, 50), 16, [300], [1], {}, "items"),                    # width not a multiple of 4
]


@pytest.mark.parametrize("window", [0, 333])
@pytest.mark.parametrize("kv,geo,bt,prior,new,opt,want", FORMS,
                         ids=[f"{f[0]}-{'x'.join(map(str, f[1]))}-bt{f[2]}-{'_'.join(map(str, f[4]))}" + ("-set" if f[5] else "")
                              for f in FORMS])
def test_route_and_cover(kv, geo, bt, prior, new, opt, want, window):
    segs, start = [], 0
    for s, (p, n) in enumerate(zip(prior, new)):
        segs.append((s, start, n, p))
        start += n
    table = contiguous_table([p + n for p, n in zip(prior, new)], bt)
    for n_cu in (256, 80, 12):
        for noalloc in (False, True):
            items, merges, units, c = plan(kv, *geo, bt, table, segs, window=window, n_cu=n_cu, noalloc=noalloc, **opt)
            check_plan(kv, *geo, bt, table, segs, window, items, merges, units, c, noalloc=noalloc)
            if n_cu != 256 or window:
                continue
            small_units = len(units) > 0 and int(units[:, 6].max()) <= 32
            got = "items" if len(units) == 0 else "units" if small_units and len(items) == 0 else "prefill"
            assert got == want, (got, len(items), len(units))
            if noalloc and got == "units":   # no partials outside the workgroups
                assert c.slots == 0 and len(merges) == 0


def test_long_units_are_cut_and_short_ones_packed():
    """One long context: its units run as key pieces that a merge launch combines; many short rows:
    whole units, no merges, and no more workgroups than the device holds at once."""
    geo = (64, 8, 128, 128)
    table = contiguous_table([9007], 16)
    segs = [(0, 0, 7, 9000)]
    items, merges, units, c = plan("f16", *geo, 16, table, segs)
    check_plan("f16", *geo, 16, table, segs, 0, items, merges, units, c)
    assert c.slots > 0 and len(merges) > 0 and len(items) == 0
    assert c.pf_wg <= 512   # 8 waves per CU: 256 workgroups of 8, or 512 of 4
    prior, new = [700 + 3 * i for i in range(32)], [3] * 32
    table = contiguous_table([p + 3 for p in prior], 16)
    segs = [(i, 3 * i, 3, p) for i, p in enumerate(prior)]
    items, merges, units, c = plan("f16", 32, 8, 128, 128, 16, table, segs)
    check_plan("f16", 32, 8, 128, 128, 16, table, segs, 0, items, merges, units, c)
    assert c.slots == 0 and len(merges) == 0 and len(items) == 0 and c.pf_wg <= 512


def test_allocation_free_calls_keep_a_list_that_fits():
    """The staging an allocation-free call may use (1 MiB here) takes 900 single rows of 32 KV heads as
    decode items, not as unit records; fewer rows, and calls that may allocate, are units."""
    geo = (32, 32, 80, 80)
    for n, noalloc, units_expected in ((900, True, False), (900, False, True), (500, True, True)):
        table = contiguous_table([21] * n, 16)
        segs = [(i, i, 1, 20) for i in range(n)]
        items, merges, units, c = plan("f16", *geo, 16, table, segs, noalloc=noalloc)
        assert (len(units) > 0) == units_expected and (len(items) > 0) != units_expected, (n, noalloc)
        if len(items):
            assert len(items) * 32 + n * 8 <= 1 << 20
        check_plan("f16", *geo, 16, table, segs, 0, items, merges, units, c, noalloc=noalloc)


def test_a_call_given_back_keeps_the_items_head_blocks():
    """Too many single rows for the staging of an allocation-free call, in a group wider than the
    row-layout kernel's 4 heads per item: its items hold 4 heads each."""
    geo, n = (128, 16, 80, 80), 1700
    table = contiguous_table([21] * n, 16)
    segs = [(i, i, 1, 20) for i in range(n)]
    items, merges, units, c = plan("f16", *geo, 16, table, segs, noalloc=True)
    assert len(units) == 0 and len(items) == n * 16 * 2 and c.ng == 4
    check_plan("f16", *geo, 16, table, segs, 0, items, merges, units, c, noalloc=True)


@pytest.mark.parametrize("kv,geo,new", [
    ("f16", (12, 2, 128, 128), 4), ("q8_0", (12, 2, 128, 128), 4), ("f16", (8, 1, 128, 128), 4), ("bf16", (8, 1, 256, 256), 6),
    ("f16", (4, 1, 80, 80), 1), ("bf16", (6, 2, 80, 80), 1), ("f32", (16, 2, 128, 128), 1), ("f32", (3, 3, 64, 64), 3)])
@pytest.mark.parametrize("ctx", [8000, 32000, 130000])
def test_few_units_share_a_long_context_evenly(kv, geo, new, ctx):
    """One sequence, one to three KV heads: a unit runs as at most 64 pieces, no piece more than twice
    the pages of an even share (of the pieces, or of 512 workgroups where those are fewer; a workgroup
    of 8 waves of 4 pages at the least). Short contexts may stay on the decode items."""
    table = contiguous_table([ctx + new], 16)
    segs = [(0, 0, new, ctx)]
    items, merges, units, c = plan(kv, *geo, 16, table, segs)
    check_plan(kv, *geo, 16, table, segs, 0, items, merges, units, c)
    assert len(units) > 0 or (ctx < 130000 and new > 1)
    n_pages = (ctx + new + 15) // 16
    live = [u for u in units if int(u[4]) != 0]
    n_units = len({(int(u[1]), int(u[5])) for u in live})
    longest = max([int(u[8]) for u in live], default=0)
    assert longest <= 2 * max(n_pages / 64, n_pages * n_units / 512) + 32, (longest, n_pages, n_units)


@pytest.mark.parametrize("kv,geo,new", [
    ("f16", (32, 8, 128, 128), 4), ("q8_0", (32, 8, 128, 128), 4), ("f16", (12, 2, 128, 128), 4), ("bf16", (16, 4, 256, 256), 4),
    ("f16", (8, 2, 80, 80), 1), ("f16", (8, 8, 80, 80), 1), ("f32", (64, 8, 128, 128), 1), ("bf16", (64, 4, 256, 256), 7)])
@pytest.mark.parametrize("ctx", [9000, 32000])
def test_allocation_free_calls_share_a_long_context_too(kv, geo, new, ctx):
    """Pieces whose partials and merges fit the scratch (check_plan), the same as a call that may
    allocate takes: no wave walks more than in that call's plan, or in decode items'."""
    table = contiguous_table([ctx + new], 16)
    segs = [(0, 0, new, ctx)]
    longest = []
    for noalloc in (False, True):
        items, merges, units, c = plan(kv, *geo, 16, table, segs, noalloc=noalloc)
        check_plan(kv, *geo, 16, table, segs, 0, items, merges, units, c, noalloc=noalloc)
        longest.append(max((int(u[8]) for u in units if int(u[4]) != 0), default=0))
        if noalloc:
            assert c.slots * c.ng * (geo[3] + 4) * 4 + 256 + len(merges) * 24 <= 32 << 20
    assert longest[1] <= 1.5 * longest[0], longest


@pytest.mark.parametrize("kv,geo,new", [
    ("bf16", (32, 1, 80, 80), 1), ("f32", (64, 2, 128, 128), 1), ("f16", (64, 2, 128, 128), 4), ("f16", (71, 1, 64, 64), 4),
    ("f32", (71, 1, 64, 64), 1), ("f16", (128, 1, 256, 256), 3)])
@pytest.mark.parametrize("noalloc", [False, True])
def test_groups_wider_than_a_unit_share_a_long_context(kv, geo, new, noalloc):
    """More heads per group than the 16 or 32 columns of a unit: the units are cut into pieces all the
    same, their partials at their head's position of a slot of the whole group."""
    ctx = 32000
    table = contiguous_table([ctx + new], 16)
    segs = [(0, 0, new, ctx)]
    items, merges, units, c = plan(kv, *geo, 16, table, segs, noalloc=noalloc)
    check_plan(kv, *geo, 16, table, segs, 0, items, merges, units, c, noalloc=noalloc)
    live = [u for u in units if int(u[4]) != 0]
    n_units = len({(int(u[1]), int(u[2]), int(u[5])) for u in live})
    n_pages = (ctx + new + 15) // 16
    assert live and c.ng == geo[0] // geo[1] and all(int(u[5]) + int(u[6]) <= c.ng * int(u[4]) for u in live)
    assert max(int(u[8]) for u in live) <= 2 * max(n_pages / 64, n_pages * n_units / 512) + 32
    if noalloc:
        assert c.slots * c.ng * (geo[3] + 4) * 4 + 256 + len(merges) * 24 <= 32 << 20


def test_whole_units_give_a_long_context_back():
    """Units never cut into pieces (prefill_whole_units): a call they would leave on a few workgroups stays
    on the decode items, one whose units fill the device does not."""
    for new, prior, units_expected in (([4], [32000], False), ([6] * 4, [2000] * 4, True), ([1], [32000], None)):
        kv, geo = ("f16", (32, 8, 128, 128)) if units_expected is not None else ("f32", (64, 2, 128, 128))
        segs, start = [], 0
        for s, (p, n) in enumerate(zip(prior, new)):
            segs.append((s, start, n, p))
            start += n
        table = contiguous_table([p + n for p, n in zip(prior, new)], 16)
        items, merges, units, c = plan(kv, *geo, 16, table, segs, prefill_whole_units=1)
        check_plan(kv, *geo, 16, table, segs, 0, items, merges, units, c)
        assert (len(units) > 0) == bool(units_expected) and (len(items) > 0) != bool(units_expected)


def wave_plan(kv, n_head, n_kv, hd, hdv, bt, table, segs, window, n_cu, per_cu, noalloc):
    n_seqs, bps = table.shape
    tab = np.ascontiguousarray(table, dtype=np.int32)
    d = N.PlanDesc(N.ABI_VERSION, KV[kv], n_head, n_kv, hd, hdv, bt, n_cu, 0, n_seqs, bps, tab.ctypes.data_as(C.c_void_p),
                   window, 0.1, int(noalloc), N.AttendTuning(N.ABI_VERSION, 0, 0, 0, 0, 0, 0, 0))
    arr = (N.Seg * len(segs))(*[N.Seg(*s) for s in segs])
    c = N.PlanWaveCounts()
    args = (C.byref(d), arr, len(segs), per_cu)
    rc = N.lib().lmh_plan_unit_waves(*args, None, 0, None, 0, C.byref(c))
    waves = np.zeros((c.n_waves, c.wave_words), np.uint32)
    merges = np.zeros((c.n_merges, c.merge_words), np.uint32)
    if rc != N.OK:
        rc = N.lib().lmh_plan_unit_waves(*args, waves.ctypes.data_as(C.c_void_p), c.n_waves,
                                         merges.ctypes.data_as(C.c_void_p), c.n_merges, C.byref(c))
    assert rc == N.OK
    return waves, merges, c


WAVE_CALLS = [(f[0], f[1], f[2], f[3], f[4]) for f in FORMS if f[6] == "units"] + [
    ("f16", (64, 8, 128, 128), 16, [9000], [7]), ("f16", (12, 2, 128, 128), 32, [30000], [4]), ("f32", (64, 2, 128, 128), 16, [9000, 5], [1, 9]),
    ("bf16", (32, 1, 80, 80), 16, [20000, 50], [1, 2]), ("q8_0", (32, 8, 128, 128), 16, [3000, 1700, 800, 40], [4, 7, 2, 5]),
    ("bf16", (16, 4, 256, 256), 64, [10, 700], [1500, 333]), ("f16", (32, 32, 80, 80), 16, [700 * i for i in range(9)], [1] * 8 + [120]),
]


@pytest.mark.parametrize("kv,geo,bt,prior,new", WAVE_CALLS,
                         ids=[f"{f[0]}-{'x'.join(map(str, f[1]))}-{'_'.join(map(str, f[4]))}" for f in WAVE_CALLS])
@pytest.mark.parametrize("window", [0, 333])
def test_wave_records(kv, geo, bt, prior, new, window):
    """The records a unit launch reads, over device sizes and occupancies: a unit's (or piece's) waves are
    consecutive in one workgroup and share its pages in order, each a whole number of steps but the last,
    with the block ids of the first two; put together they are a plan that covers every row once."""
    segs, start = [], 0
    for s, (p, n) in enumerate(zip(prior, new)):
        segs.append((s, start, n, p))
        start += n
    table = contiguous_table([p + n for p, n in zip(prior, new)], bt)
    step = 1 if kv == "f32" else 2
    for n_cu, per_cu in ((256, 4), (256, 8), (256, 12), (256, 16), (80, 8), (12, 8), (5, 4)):
        for noalloc in (False, True):
            waves, merges, c = wave_plan(kv, *geo, bt, table, segs, window, n_cu, per_cu, noalloc)
            if not len(waves):
                continue   # given back to the items
            W, units, at = c.waves_per_wg, [], 0
            assert len(waves) % W == 0
            while at < len(waves):
                seq, row0, pos0, page0, n_pages, slot, b0, b1, head, cols = (int(x) for x in waves[at])
                n = cols >> 16 & 0xFF
                if n == 0:
                    assert not waves[at].any()
                    at += 1
                    continue
                assert at // W == (at + n - 1) // W and (n == 1 or c.shared)
                page = page0
                for j in range(n):
                    r = [int(x) for x in waves[at + j]]
                    assert (r[0], r[1], r[2], r[5], r[8]) == (seq, row0, pos0, slot, head)
                    assert r[9] == (cols & ~0xFF00) | j << 8
                    assert r[3] == page and r[4] > 0 and (j + 1 == n or r[4] % step == 0)
                    assert r[6] == table[seq, page * 16 // bt] and r[7] == table[seq, min(page + 1, page + r[4] - 1) * 16 // bt]
                    page += r[4]
                kvh, c_off, n_col, k = head & 0xFFFF, head >> 16, cols & 0xFF, cols >> 24
                assert n_col <= 16 * c.col_blocks and (k > 1) == (slot != NO_SLOT)
                n_tok = (c_off + n_col - 1) // (geo[0] // geo[1]) + 1
                total = page - page0
                units.append([seq, kvh, row0, pos0, n_tok, c_off, n_col, page0, total, slot, k, 0] +
                             [int(table[seq, (page0 + min(b, total - 1)) * 16 // bt]) for b in range(8)])
                at += n
            counts = SimpleNamespace(ng=c.ng, slots=c.slots, pf_wg=len(units), pf_per_wg=1, max_pages=1 << 30, local=0,
                                     layout=c.layout, chunk=0)
            check_plan(kv, *geo, bt, table, segs, window, np.zeros((0, 8), np.uint32), merges, np.array(units), counts,
                       noalloc=noalloc)
