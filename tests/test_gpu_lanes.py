"""One lane per pair (k_align_lanes) against the oracle, at the LCS level and
tile by tile: every window width it holds, targets at both ends of each width's
lengths, unknown letters, shifted and unrelated targets.  NGIA_LANE_FILL=0
sends every window of up to 40 words there, whatever the bin's size."""
import os

import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from conftest import AMINO, mutate
from test_gpu_parity import expected_run_tiles, say

pytestmark = pytest.mark.gpu
LANE_MAX = 40


def lane_pairs(rng, identity):
    """(records, lengths, jobs): per width, reps with related, shifted,
    low-complexity and partly unknown targets of the shortest, a middle and the
    longest length that give the width."""
    thr = float(np.float32(identity) / np.float32(100))
    by_w = {}
    step = 1 if identity <= 60 else 3
    for T in range(1, 6500, step):
        for R in {T, T + 7, int(T / thr), (T + 31) // 32 * 32}:
            if R < T or np.float32(T) < np.float32(R) * np.float32(thr):
                continue
            by_w.setdefault(orc.band_window(R, T, thr), []).append((R, T))
        if min(by_w) > LANE_MAX:
            break
    seqs, jobs = [], []
    for W in range(2, LANE_MAX + 1):
        c = sorted(by_w.get(W, []))
        for R, T in {c[0], c[len(c) // 2], c[-1]} if c else ():
            anc = bytes(AMINO[i] for i in rng.integers(20, size=R))
            sh = max(1, int(R * (1 - thr)) // 2)
            low = bytearray(b"A" * T)
            for p in rng.integers(0, T, size=max(1, T // 40)):
                low[p] = AMINO[int(rng.integers(1, 20))]
            unk = bytearray(anc[:T])
            for p in rng.integers(0, T, size=max(1, T // 10)):
                unk[p] = ord("X")
            rx = bytearray(anc)
            for p in rng.integers(0, R, size=max(1, R // 10)):
                rx[p] = ord("X")
            tars = [mutate(rng, anc[:T], 0.05, 0.0), (anc[sh:] + anc[:sh])[:T], bytes(low), bytes(unk)]
            for rep in (anc, bytes(rx)):
                r = len(seqs)
                seqs.append(rep)
                for t in tars:
                    jobs.append((r, len(seqs)))
                    seqs.append(t)
    recs = [orc.pack(s) for s in seqs]
    off = np.cumsum([0] + [len(x) for x in recs[:-1]]).astype(np.uint64)
    rep = np.arange(len(seqs), dtype=np.uint32)
    for r, t in jobs:
        rep[t] = r
    return recs, np.concatenate(recs).astype(np.uint32), off, \
        np.array([len(s) for s in seqs], dtype=np.uint32), rep.reshape(1, -1)


def context(**env):
    os.environ.update({k: str(v) for k, v in env.items()})
    try:
        return ng.Context(0)
    finally:
        for k in env:
            del os.environ[k]


@pytest.mark.parametrize("identity", [30, 50, 90])
def test_lanes_every_width(identity):
    rng = np.random.default_rng(identity)
    recs, packed, off, lengths, rep = lane_pairs(rng, identity)
    thr = float(np.float32(identity) / np.float32(100))
    for raw in (True, False):
        say("lanes, identity", identity, "records", len(recs), "raw lcs", raw)
        with context(NGIA_LANE_FILL=0, **({"NGIA_RAW_LCS": 1} if raw else {})) as c:
            db = ng.Database(c, packed, off, lengths)
            db.set_reps(rep, 1)
            db.graph(identity, 1, ng.GRAPH_BATCHED if raw else ng.GRAPH_BATCHED_TALLY)
            keys, sc = db.pair_scores()
            jobs = np.zeros((len(keys), 3), dtype=np.uint32)
            jobs[:, 0] = keys >> np.uint64(32)
            jobs[:, 1] = keys & np.uint64(0xFFFFFFFF)
            want = orc.align_jobs(packed, off, jobs, thr, raw_lcs=raw)
            np.testing.assert_array_equal(sc, want[:, 2])
            bins = {(b["kind"], b["width"]): b["run_tiles"] for b in db.bin_stats() if b["pairs"]}
            assert {k for k, _ in bins} == {"window"}
            assert {w for _, w in bins} >= set(range(3, LANE_MAX + 1))
            if not raw:
                tiles = {}
                for u, v in jobs[:, :2]:
                    R, T = int(lengths[u]), int(lengths[v])
                    lcs, t = orc.align_blocks(recs[u], recs[v], thr)
                    W = orc.band_window(R, T, thr)
                    key = ("window", W)
                    tiles[key] = tiles.get(key, 0) + expected_run_tiles(R, T, thr, lcs, t,
                                                                        W if W <= 16 else 2)
                assert bins == tiles
            db.close()
