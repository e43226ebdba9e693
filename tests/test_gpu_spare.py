"""Calls whose workspace the device refuses: NGIA_SPARE_LIMIT makes the
allocations that a call can do without fail past a size, and the call then takes
the form that needs less memory, with the same results."""
import os

import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from conftest import AMINO, mutate
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


def limited(limit):
    os.environ["NGIA_SPARE_LIMIT"] = str(limit)
    try:
        return ng.Context(0)
    finally:
        del os.environ["NGIA_SPARE_LIMIT"]


def long_set():
    """Four relatives of 40,000 residues: windows past the widest wavefront
    kernel's at -i 10."""
    rng = np.random.default_rng(3)
    anc = bytes(AMINO[i] for i in rng.integers(20, size=40000))
    seqs = [anc] + [mutate(rng, anc, 0.05, 0.0) for _ in range(3)]
    packed, off = orc.pack_many(seqs)
    return packed, off, np.array([len(s) for s in seqs], dtype=np.uint32)


@pytest.mark.parametrize("limit", [0, 1 << 20])  # all of it; the widest windows' part
def test_align(limit):
    packed, off, _ = long_set()
    jobs = np.array([(i % 4, i // 4 % 4, 0) for i in range(16)], dtype=np.uint32)
    want = orc.align_jobs(packed, off, jobs, 0.1)
    assert (want[:, 2] > 0).all()
    say("align without its workspace", limit)
    with limited(limit) as c:
        for _ in range(2):
            np.testing.assert_array_equal(c.align(packed, off, jobs, 0.1), want)


def plain_fast(c, packed, off, lengths, rep, bands, identity):
    db = ng.Database(c, packed, off, lengths)
    db.set_reps(rep, 64)
    got, tot = db.fast(identity, bands)
    again, tot2 = db.fast(identity, bands)
    db.close()
    want, wtot = orc.fast_cluster(packed, off, lengths, rep, bands, identity)
    assert tot == tot2 == wtot
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(again, want)
    return want


@pytest.mark.parametrize("cfg,scale,identity,bands", [(1, 0.1, 50, 64), (1, 0.1, 95, 64), (2, 0.052, 85, 17),
                                                      (4, 0.005, 90, 64), (3, 0.002, 97, 64), (1, 0.1, 70, 1)])
def test_fast_band_by_band(cfg, scale, identity, bands):
    d = ng.gen_packed(ng.gen_config(cfg, scale, 5))
    rep = orc.bucket(orc.sketch_all(d.packed, d.word_off))
    say("fast mode band by band, config", cfg, scale, "identity", identity, "bands", bands)
    with limited(0) as c:
        plain_fast(c, d.packed, d.word_off, d.lengths, rep, bands, identity)


@pytest.mark.parametrize("limit", [0, 1 << 20])
def test_fast_long(limit):
    packed, off, lengths = long_set()
    rep = np.tile(np.maximum(np.arange(4, dtype=np.int64) - 1, 0).astype(np.uint32), (64, 1))
    say("fast mode without its workspace", limit)
    with limited(limit) as c:
        want = plain_fast(c, packed, off, lengths, rep, 8, 10)
    assert (want == 0).all()


def test_fast_workspace_is_given_back():
    """An allocation that fails takes back what fast calls of other databases
    keep: 100,000 records' pair lists of 130 MB."""
    n = 100000
    rng = np.random.default_rng(2)
    packed, off = orc.pack_many([bytes(AMINO[i] for i in rng.integers(20, size=16)) for _ in range(1000)])
    off = np.tile(off, n // 1000)
    rep = np.tile(np.maximum(np.arange(n, dtype=np.int64) - 1000, 0).astype(np.uint32), (64, 1))
    jobs = np.zeros((3000000, 3), dtype=np.uint32)
    say("fast workspace given back")
    with limited(52 << 20) as c:
        db = ng.Database(c, packed, off)
        db.set_reps(rep, 64)
        first, _ = db.fast(90)
        held = c.info()["hbm_free"]
        assert (c.align(packed, off[:1], jobs, 0.9)[:, 2] == 100).all()
        assert c.info()["hbm_free"] > held + (100 << 20)
        again, _ = db.fast(90)
        db.close()
    np.testing.assert_array_equal(again, first)


@pytest.mark.parametrize("letters,n,L", [(AMINO, 16385, 60), (AMINO, 20000, 60), (b"ACGT", 16385, 400)])
def test_bucket_and_step(letters, n, L):
    rng = np.random.default_rng(n)
    aa = np.frombuffer(letters, dtype=np.uint8)
    anc = aa[rng.integers(0, len(aa), size=(n // 20 + 1, L))]
    seqs = anc[np.arange(n) // 20]
    sub = rng.random(seqs.shape) < 0.03
    seqs[sub] = aa[rng.integers(0, len(aa), size=int(sub.sum()))]
    packed, off = orc.pack_many([s.tobytes() for s in seqs])
    lengths = np.full(n, L, dtype=np.uint32)
    sig = orc.sketch_all(packed, off)
    rep = orc.bucket(sig)
    want, _ = orc.build_graph(packed, off, lengths, rep, 64, 90)
    say("bucketing without the partitions' room", letters[:4], n)
    with limited(0) as c:
        np.testing.assert_array_equal(c.bucket(sig), rep)
        db = ng.Database(c, packed, off, lengths)
        db.sketch()
        db.bucket()
        np.testing.assert_array_equal(db.reps(), rep)
        db.step(90)
        np.testing.assert_array_equal(db.reps(), rep)
        np.testing.assert_array_equal(db.edges(), want)
        db.close()
