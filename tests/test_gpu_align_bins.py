"""The align call through the length bins, against the oracle: job counts on
both sides of the plain kernel's, targets shorter and longer than the rep,
residues and DNA, thresholds that no bin is made for."""
import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from conftest import AMINO, mutate

pytestmark = pytest.mark.gpu


def records(seed, letters, lo, hi, count):
    rng = np.random.default_rng(seed)
    seqs = []
    for _ in range(count // 4):
        L = int(np.exp(rng.uniform(np.log(lo), np.log(hi))))
        anc = bytes(letters[i] for i in rng.integers(len(letters), size=L))
        seqs += [anc, mutate(rng, anc, 0.03, 0.01), anc[: max(1, L * 3 // 4)], anc[L // 9:]]
    return seqs + [b"", b"A"]


@pytest.mark.parametrize("letters", [AMINO, b"ACGT"])
@pytest.mark.parametrize("thr", [0.01, 0.2, 0.5, 0.7, 0.9, 0.99])
@pytest.mark.parametrize("count", [1, 15, 16, 17, 3000, 6000])
def test_jobs(ctx, letters, thr, count):
    seqs = records(int(thr * 100) + count, letters, 8, 1500, 120)
    packed, off = orc.pack_many(seqs)
    rng = np.random.default_rng(count)
    n = len(seqs)
    jobs = np.zeros((count, 3), dtype=np.uint32)
    jobs[:, 0] = rng.integers(0, n, count)
    jobs[:, 1] = rng.integers(0, n, count)
    near = rng.random(count) < 0.5  # the same ancestor's
    jobs[near, 1] = jobs[near, 0] // 4 * 4 + rng.integers(0, 4, near.sum())
    jobs[:, 1] %= n
    print("align jobs", letters[:4], thr, count, flush=True)
    want = orc.align_jobs(packed, off, jobs, thr)
    np.testing.assert_array_equal(ctx.align(packed, off, jobs, thr), want)
    assert count < 3000 or (want[:, 2] > 0).any()


@pytest.mark.parametrize("length", [3000, 20000, 65534])
def test_long_records(ctx, length):
    """Windows up to the widest wavefront kernel's and past it."""
    rng = np.random.default_rng(length)
    anc = bytes(AMINO[i] for i in rng.integers(20, size=length))
    seqs = [anc, mutate(rng, anc, 0.05, 0.0), anc[: length // 2], anc[: length // 3]]
    packed, off = orc.pack_many(seqs)
    jobs = np.array([(i % 4, i // 4 % 4, 0) for i in range(64)], dtype=np.uint32)
    for thr in (0.3, 0.9):
        print("align long", length, thr, flush=True)
        np.testing.assert_array_equal(ctx.align(packed, off, jobs, thr),
                                      orc.align_jobs(packed, off, jobs, thr))


@pytest.mark.parametrize("thr", [0.0, 1.0, 1.25])
def test_other_thresholds(ctx, thr):
    seqs = records(5, AMINO, 8, 400, 80)
    packed, off = orc.pack_many(seqs)
    rng = np.random.default_rng(7)
    jobs = np.zeros((500, 3), dtype=np.uint32)
    jobs[:, :2] = rng.integers(0, len(seqs), (500, 2))
    print("align threshold", thr, flush=True)
    np.testing.assert_array_equal(ctx.align(packed, off, jobs, thr),
                                  orc.align_jobs(packed, off, jobs, thr))


@pytest.mark.parametrize("count", [1, 15, 16, 17, 400])
@pytest.mark.parametrize("thr", [0.0, 0.7, 1.0, 1.25])
def test_score_column_is_overwritten(ctx, count, thr):
    """Whatever the third column holds, a job that the length filter rejects
    scores 0, like any other that does not pass."""
    seqs = records(9, AMINO, 8, 400, 80)
    packed, off = orc.pack_many(seqs)
    rng = np.random.default_rng(count)
    jobs = np.zeros((count, 3), dtype=np.uint32)
    jobs[:, :2] = rng.integers(0, len(seqs), (count, 2))
    jobs[0, :2] = 0, len(seqs) - 1  # a single residue
    want = orc.align_jobs(packed, off, jobs, thr)
    jobs[:, 2] = 77
    print("align with an old score column", count, thr, flush=True)
    np.testing.assert_array_equal(ctx.align(packed, off, jobs, thr), want)


@pytest.mark.parametrize("lengths", [(500,), (60, 500), (60, 500, 1100), (60, 500, 1100, 2400),
                                     (60, 300, 500, 800, 1100, 1900, 2400, 5200)])
def test_one_to_many_kernels(ctx, lengths):
    """A call whose jobs one kernel aligns runs on one stream, others on as many
    side streams as kernels; calls in a row, each waiting for the one before."""
    rng = np.random.default_rng(len(lengths))
    seqs = []
    for L in lengths:
        anc = bytes(AMINO[i] for i in rng.integers(20, size=L))
        seqs += [anc] + [mutate(rng, anc, 0.04, 0.01)[:L] for _ in range(3)]
    packed, off = orc.pack_many(seqs)
    for count in (16, 200, 7000):
        jobs = np.zeros((count, 3), dtype=np.uint32)
        jobs[:, 0] = rng.integers(0, len(seqs), count)
        jobs[:, 1] = jobs[:, 0] // 4 * 4 + rng.integers(0, 4, count)
        for thr in (0.5, 0.8):
            print("align streams", lengths, count, thr, flush=True)
            want = orc.align_jobs(packed, off, jobs, thr)
            assert (want[:, 2] > 0).any()
            for _ in range(2):
                np.testing.assert_array_equal(ctx.align(packed, off, jobs, thr), want)
