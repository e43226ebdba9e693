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

