"""The batched fast mode against the oracle's band-by-band clustering: one round
and two (split at 50,000 records), DNA, fewer bands than rows, a set without
candidates; the last graph's pairs and edges stay as they were."""
import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc
from test_gpu_parity import say

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("cfg,scale,identity,bands", [(1, 0.1, 50, 64), (1, 0.1, 95, 64), (2, 0.052, 60, 64),
                                                      (2, 0.052, 85, 17), (2, 0.052, 85, 16),
                                                      (4, 0.005, 90, 64), (3, 0.002, 97, 64),
                                                      (1, 0.1, 70, 1)])
def test_fast_batched(ctx, cfg, scale, identity, bands):
    say("fast mode, config", cfg, scale, "identity", identity, "bands", bands)
    d = ng.gen_packed(ng.gen_config(cfg, scale, 5))
    db = ng.Database(ctx, d.packed, d.word_off, d.lengths)
    db.sketch()
    db.bucket()
    rep = db.reps()
    db.graph(identity, bands)
    edges, (keys, sc) = db.edges(), db.pair_scores()
    got, tot = db.fast(identity, bands)
    want, wtot = orc.fast_cluster(d.packed, d.word_off, d.lengths, rep, bands, identity)
    assert tot == wtot
    np.testing.assert_array_equal(got, want)
    np.testing.assert_array_equal(db.edges(), edges)
    keys2, sc2 = db.pair_scores()
    np.testing.assert_array_equal(keys2, keys)
    np.testing.assert_array_equal(sc2, sc)
    db.graph(identity, bands)
    np.testing.assert_array_equal(db.edges(), edges)
    db.close()


def test_fast_without_candidates(ctx):
    d = ng.gen_packed(ng.gen_config(1, 0.02, 5))
    db = ng.Database(ctx, d.packed, d.word_off, d.lengths)
    db.set_reps(np.tile(np.arange(d.n, dtype=np.uint32), (64, 1)), 64)
    got, tot = db.fast(90)
    assert tot == 0
    np.testing.assert_array_equal(got, np.arange(d.n))
    db.close()
