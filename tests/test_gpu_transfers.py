"""Rows to the device and back at the sizes where the transfers change: below
and from 4 MiB on, slots of 2 MiB filled and started, all four and more."""
import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n", [1, 8192, 16383, 16384, 16385, 24577, 32767, 32768, 32769, 50001])
def test_rows_there_and_back(ctx, n):
    packed, off = orc.pack_many([b"ACDEFGHIKL"] * n)
    db = ng.Database(ctx, packed, off)
    rng = np.random.default_rng(n)
    print("rows of", n, flush=True)
    for _ in range(3):
        rows = rng.integers(0, n, size=(64, n), dtype=np.uint64).astype(np.uint32)
        db.set_reps(rows, 64)
        np.testing.assert_array_equal(db.reps(), rows)
    rows[63, n - 1] = n
    with pytest.raises(ng.NgiaError):
        db.set_reps(rows, 64)
    db.close()
