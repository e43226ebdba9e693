"""The four-letter sketch (k_sketch_walk) against the oracle: databases of four
letters, of three, and of five with N among them; records short and long, of few
different 8-mers, with runs of unknown letters, and of lengths around the
blocks of 32 and the bound below which every window is hashed."""
import os

import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def records(rng, alpha, odd):
    seqs = []

    def rand(L):
        return bytearray(alpha[i] for i in rng.integers(len(alpha), size=L))

    for L in (0, 1, 7, 8, 9, 100, 400, 440, 442, 443, 444, 445, 450, 479, 480, 481, 1000, 2047, 2048,
              2049, 2055, 2056, 4096, 30000, 65534):
        seqs.append(rand(L))
    for L in (500, 3000, 60000):  # few different 8-mers
        seqs.append(bytearray(alpha[:1] * L))
        seqs.append(bytearray((alpha[:2] * L)[:L]))
        unit = rand(50)
        seqs.append((unit * (L // 50 + 1))[:L])
    for L in (600, 1400, 5000):  # rarer letters: one, a run, a tenth, everywhere
        for k in (1, 40, L // 10, L):
            s = rand(L)
            for p in rng.integers(0, L, size=k):
                s[p] = odd[int(rng.integers(len(odd)))]
            seqs.append(s)
    for p in (0, 6, 7, 8, 31, 32, 33, 39, 599):  # one other letter near a block's edge
        s = rand(600)
        s[p] = odd[0]
        seqs.append(s)
    while sum(map(len, seqs)) < 4500000:
        seqs.append(rand(int(rng.integers(200, 3000))))
    return [bytes(s) for s in seqs]


@pytest.mark.parametrize("alpha,odd", [(b"ACGT", b"X"), (b"ACGT", b"N"), (b"ACGT", b"NX"), (b"ACG", b"X")])
def test_walk_matches_oracle(ctx, alpha, odd):
    say("four-letter sketch", alpha, odd)
    rng = np.random.default_rng(len(alpha) + 10 * odd[0] + len(odd))
    recs = [orc.pack(s) for s in records(rng, alpha, odd)]
    off = np.cumsum([0] + [len(r) for r in recs[:-1]]).astype(np.uint64)
    packed = np.concatenate(recs).astype(np.uint32)
    want = orc.sketch_all(packed, off)
    db = ng.Database(ctx, packed, off)
    for _ in range(2):
        db.sketch()
        np.testing.assert_array_equal(db.sigs(), want)
    db.close()
    np.testing.assert_array_equal(ctx.sketch(packed, off), want)


def test_bits_past_a_record(ctx):
    """A signature ends with its record, whatever the last block's planes hold
    past it."""
    rng = np.random.default_rng(4)
    seqs = [bytes(b"ACGT"[i] for i in rng.integers(4, size=int(L)))
            for L in list(range(1377, 1412)) + list(rng.integers(400, 60000, size=150))]
    recs = [orc.pack(s) for s in seqs]
    off = np.cumsum([0] + [len(r) for r in recs[:-1]]).astype(np.uint64)
    want = orc.sketch_all(np.concatenate(recs).astype(np.uint32), off)
    assert sum(map(len, seqs)) > 4000000
    for s, r in zip(seqs, recs):
        left = len(s) % 32
        for p in range(4 * (left > 0)):  # the codes before, again
            r[-4 + p] |= (int(r[-8 + p]) >> left << left) & 0xFFFFFFFF
    packed = np.concatenate(recs).astype(np.uint32)
    say("four-letter sketch with bits past the records")
    np.testing.assert_array_equal(ctx.sketch(packed, off), want)


@pytest.mark.parametrize("alpha,odd", [(b"ACGT", b"NX"), (b"ACGTN", b"X")])
def test_step_with_records_of_both_forms(alpha, odd):
    """Records too short, of too many other letters or of five letters are
    hashed window by window, the others walk; a step's head comes off the front of
    both lists."""
    rng = np.random.default_rng(len(alpha))
    seqs = [bytes(alpha[i] for i in rng.integers(len(alpha), size=L)) for L in range(12000, 12020)]
    seqs += [odd[:1] * 11500] + [odd[-1:] * 60 + s[:10500] for s in seqs[:3]]
    seqs = sorted(seqs + records(rng, alpha, odd)[30:], key=len, reverse=True)
    packed, off = orc.pack_many(seqs)
    lengths = np.array([len(s) for s in seqs], dtype=np.uint32)
    want = orc.sketch_all(packed, off)
    os.environ["NGIA_HEAD_MIN"] = "8"
    try:
        c = ng.Context(0)
    finally:
        del os.environ["NGIA_HEAD_MIN"]
    say("four-letter sketch of a step with both forms", alpha, odd)
    with c:
        db = ng.Database(c, packed, off, lengths)
        db.step(90)
        assert c.timing()["step_head"] >= 8
        np.testing.assert_array_equal(db.sigs(), want)
        np.testing.assert_array_equal(db.reps(), orc.bucket(want))
        db.close()
