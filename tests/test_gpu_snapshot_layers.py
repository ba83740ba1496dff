"""Snapshots of several layers (write_seq / read_seq, crates/engine/model/src/kv.rs:1030-1130): runs of
layers of one geometry (a launch each) beside layers of others, granule and segment copies at widths
whose rows are whole 16-byte words, whole 4-byte words or neither, blocks above and below a tile; bytes
against the reference-format oracle, and read into blocks that held other rows before (read_seq does not
zero them: every byte is the snapshot's)."""

import numpy as np
import pytest

from test_gpu_snapshot import step, twin

pytestmark = pytest.mark.gpu

A, B, C = (8, 2, 128, 128), (4, 4, 64, 64), (4, 2, 256, 256)
CASES = [
    ("f16", [A, A, A, B, B, A], 16), ("bf16", [B, B, C, C], 32), ("q8_0", [A, A, B, C, C, C], 16),
    ("f16", [A] * 5, 64), ("q8_0", [B] * 4, 32),
    ("f32", [B, B, A], 16), ("f32", [(4, 2, 100, 36), (4, 2, 100, 36)], 32), ("f32", [(2, 1, 6, 6)] * 2, 8),
    ("f16", [(8, 2, 80, 80)] * 3 + [(4, 2, 50, 50)] * 2, 16),     # 16- and 4-byte words
    ("bf16", [(4, 2, 33, 35)] * 2, 16),                           # rows of 66 and 70 bytes: neither
    ("f16", [(1, 1, 33, 34), (1, 1, 34, 34), (1, 1, 33, 34)], 1), # rows of 68 bytes, 134 bytes into the block
    ("f16", [(1, 1, 33, 34), (1, 1, 33, 33), (1, 1, 34, 34)], 2), # blocks of 804 bytes: unwritten slots zero to the end
    ("bf16", [(1, 1, 33, 34)], 4), ("f32", [(1, 1, 5, 6)], 2), ("f16", [(1, 1, 1, 2)], 2),
    ("f16", [(8, 2, 64, 128), (8, 2, 64, 128)], 16), ("bf16", [(8, 2, 128, 128)] * 2, 4),
    ("q8_0", [(4, 2, 96, 32)] * 2, 16), ("f16", [(12, 4, 96, 96)] * 2, 16),
]


@pytest.mark.parametrize("kv,layers,bt", CASES, ids=[f"{c[0]}-{len(c[1])}x{c[1][0][2]}-bt{c[2]}" for c in CASES])
def test_layers_round_trip(cuda, kv, layers, bt):
    import torch

    rng = np.random.default_rng(17)
    hc, oc = twin(kv, n_seqs=3, max_ctx=160, bt=bt, layers=layers)
    step(hc, oc, [(0, 77), (1, 130)], rng, layers)
    snap = oc.write_seq(0)
    got = hc.write_seq(0)
    assert np.array_equal(got.cpu().numpy(), snap)
    hc.clear(1)                                   # its blocks, full of other rows, are the next ones taken
    for s in (2, 1):
        hc.read_seq(s, 77, torch.from_numpy(snap).cuda())
        assert np.array_equal(hc.write_seq(s).cpu().numpy(), snap), s
    one = twin(kv, n_seqs=1, max_ctx=160, bt=bt, layers=layers)[0]   # into a cache as it was created
    one.read_seq(0, 77, torch.from_numpy(snap).cuda())
    assert np.array_equal(one.write_seq(0).cpu().numpy(), snap)
