"""The sorted edge list of a batched round, against the oracle: no edges, one
edge, many per record, and a record with as many edges as the ranking takes,
one more and many more (rows given by the caller: every record below a star's
head), which the sort takes."""
import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from conftest import AMINO, mutate

pytestmark = pytest.mark.gpu


def database(n, seed, length=60):
    """Close copies of one ancestor, longest first."""
    rng = np.random.default_rng(seed)
    anc = bytes(AMINO[i] for i in rng.integers(20, size=length))
    seqs = sorted((mutate(rng, anc, 0.03, 0.005) for _ in range(n)), key=len, reverse=True)
    packed, off = orc.pack_many(seqs)
    return packed, off, np.array([len(s) for s in seqs], dtype=np.uint32)


@pytest.mark.parametrize("edges", [0, 1, 63, 64, 1023, 1024, 1025, 1026, 5000])
def test_star(ctx, edges):
    n = edges + 40
    packed, off, lengths = database(n, edges + 1)
    rep = np.tile(np.arange(n, dtype=np.uint32), (64, 1))
    rng = np.random.default_rng(edges)
    tars = rng.permutation(np.arange(1, n))[:edges]
    rep[rng.integers(0, 64, edges), tars] = 0  # the star's rays, each in some band
    rep[5, n - 20:] = n - 30 + (np.arange(20, dtype=np.uint32) // 4)  # and a few more heads
    want, tot = orc.build_graph(packed, off, lengths, rep, 64, 50)
    print("star of", edges, len(want), flush=True)
    db = ng.Database(ctx, packed, off, lengths)
    db.set_reps(rep, 64)
    for mode in (ng.GRAPH_BATCHED, ng.GRAPH_BATCHED, ng.GRAPH_BATCHED_EAGER):
        st = db.graph(50, 64, mode)
        np.testing.assert_array_equal(db.edges(), want)
        assert st["n_edges"] == len(want) and st["total_pairs"] == tot
    db.close()


@pytest.mark.parametrize("n", [1, 2, 255, 1023, 1024, 1025, 4095, 4096, 4097, 16384, 16385, 16390])
def test_sizes(ctx, n):
    """Rows of the bucketing itself: every record has up to 64 edges; the prefix
    sums' tiles of 4,096 and their forms on either side of 16,384."""
    packed, off, lengths = database(n, n)
    print("edge list", n, flush=True)
    rep = orc.bucket(orc.sketch_all(packed, off))
    want, _ = orc.build_graph(packed, off, lengths, rep, 64, 80)
    db = ng.Database(ctx, packed, off, lengths)
    db.step(80, 64)
    np.testing.assert_array_equal(db.edges(), want)
    db.close()


@pytest.mark.parametrize("n", [3, 60, 76, 77, 90])
@pytest.mark.parametrize("length", [60, 300])
def test_few_pairs(n, length):
    """Rounds on both sides of 3,072 pairs (rows that pair each record with up to
    64 before it): a wavefront each, or the usual shapes."""
    packed, off, lengths = database(n, n, length)
    rep = np.array([[max(i - 1 - b, 0) for i in range(n)] for b in range(64)], dtype=np.uint32)
    want, tot = orc.build_graph(packed, off, lengths, rep, 64, 60)
    print("few pairs", n, length, flush=True)
    c = ng.Context(0)
    db = ng.Database(c, packed, off, lengths)
    db.set_reps(rep, 64)
    st = db.graph(60, 64)
    np.testing.assert_array_equal(db.edges(), want)
    kinds = {b["kind"] for b in db.bin_stats() if b["pairs"]}
    few = st["distinct_pairs"] <= 3072 and length == 300
    assert ("wave" in kinds) == few
    db.close()
    c.close()


def test_database_on_another_context(ctx):
    """A round captured on one context and asked for on another: its bin counts
    reach the caller's."""
    d = ng.gen_packed(ng.gen_config(1, 0.1, 5))
    rep = orc.bucket(orc.sketch_all(d.packed, d.word_off))
    want, _ = orc.build_graph(d.packed, d.word_off, d.lengths, rep, 64, 70)
    print("one database, two contexts", flush=True)
    with ng.Context(0) as other:
        db = ng.Database(ctx, d.packed, d.word_off, d.lengths)
        db.set_reps(rep, 64)
        launches = []
        for c in (ctx, other, ctx, other):
            db.ctx = c
            launches.append(db.graph(70)["align_launches"])
            np.testing.assert_array_equal(db.edges(), want)
        db.ctx = ctx
        db.close()
    assert launches[0] > 0 and launches == launches[:1] * 4
