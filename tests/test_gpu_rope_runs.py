"""Aligned runs of four rows on q8_0 and f32 pages (qk_rope_store's slot kernel) against the oracle
(per_head_norm, rope, store: crates/engine/model/src/forward.rs:427-453): each width, both pairings,
odd head counts, norms on each kind, runs beside unaligned edges and single rows, block sizes above a
tile; and without norm or rotation the same page bytes as the rows stored one by one."""

import numpy as np
import pytest

from llmario_amd.kv import HipKvCache, Layer
from test_gpu_rope import check_case

pytestmark = pytest.mark.gpu

CASES = [
    # kv,   n_head, n_kv, hd, hdv, rot, neox,  q_norm, k_norm, v_norm, q_stride, div,   theta
    ("q8_0", 8, 2, 64, 64, 64, True, True, True, True, 0, False, 1e4),
    ("q8_0", 9, 3, 128, 128, 128, True, True, True, True, 0, False, 1e6),
    ("q8_0", 6, 3, 128, 128, 128, False, False, True, False, 256, True, 1e4),
    ("q8_0", 4, 1, 256, 256, 256, True, True, False, True, 0, False, 1e6),
    ("q8_0", 4, 2, 256, 256, 64, False, True, True, False, 0, False, 1e4),
    ("f32", 6, 3, 64, 64, 64, True, True, True, True, 0, True, 1e4),
    ("f32", 8, 2, 128, 128, 32, False, False, True, False, 0, False, 1e6),
    ("f32", 3, 1, 256, 256, 256, True, True, True, True, 0, False, 1e4),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-h{c[1]}x{c[2]}-hd{c[3]}-{'neox' if c[6] else 'norm'}")
def test_runs_match_the_oracle(cuda, case):
    check_case(case, 300 + CASES.index(case), [0, 1, 1000, 14], [(0, 38), (1, 9), (2, 4), (3, 1)], 2048)


# 256-wide heads on f32 pages take runs whole from 128 rows on; partly rotated Neox pairs sit in different
# lanes of the slot kernel, so calls of 1,024 rows or more on q8_0 and f32 pages take the row kernel of the
# register path (each row's heads in one workgroup), at each of its widths
LONG = [
    (("f32", 3, 1, 256, 256, 256, True, True, True, True, 0, False, 1e4), 150),
    (("q8_0", 8, 2, 64, 64, 32, True, True, True, False, 0, False, 1e4), 1030),
    (("f32", 8, 2, 128, 128, 64, True, False, True, True, 0, True, 1e6), 1030),
    (("q8_0", 4, 2, 256, 256, 128, True, True, False, True, 0, False, 1e6), 1030),
]


@pytest.mark.parametrize("case,n", LONG, ids=lambda c: f"{c[0]}-hd{c[3]}-rot{c[5]}" if isinstance(c, tuple) else str(c))
def test_long_calls_match_the_oracle(cuda, case, n):
    check_case(case, 400 + n, [0, 500, 0], [(0, n), (1, 3), (2, 1)], 2048)


@pytest.mark.parametrize("kv,hd,bt", [("q8_0", 64, 16), ("q8_0", 128, 32), ("q8_0", 256, 16), ("f32", 128, 64)])
def test_runs_store_the_bytes_single_rows_store(cuda, kv, hd, bt):
    import torch

    n, nh, nk = 40, 4, 3
    rng = np.random.default_rng(31)
    dev = lambda *s: torch.from_numpy(rng.standard_normal(s).astype(np.float32)).cuda()
    q, k, v = dev(n, nh, hd), dev(n, nk, hd), dev(n, nk, hd)
    k[3, 1, :32] = 0          # an all-zero q8_0 block
    v[5, 2, 32:64] = 0
    snaps = []
    for one_by_one in (False, True):
        hc = HipKvCache([Layer(nh * nk, nk, hd, hd)], max_ctx=64, n_seqs=1, kv_type=kv, block_tokens=bt)
        hc.reserve(0, n)
        qq = q.repeat(1, nk, 1)
        out = torch.empty_like(qq)
        for i in range(0, n, 1 if one_by_one else n):
            m = 1 if one_by_one else n
            hc.qk_rope_store(0, [(0, 0, m, i)], qq[i:i + m].contiguous(), k[i:i + m].contiguous(), v[i:i + m].contiguous(),
                             out[i:i + m], rope=False)
        hc.set_len(0, n)
        snaps.append((hc.write_seq(0).cpu().numpy(), out.cpu().numpy()))
    assert np.array_equal(snaps[0][1], snaps[1][1])
    assert np.array_equal(snaps[0][0], snaps[1][0])
