"""The partitioned bucketing at its edges, against the oracle's stable sort:
record counts at the partition counts' steps and at the tiles of the scatter,
signatures repeated past a chain's length, past a partition's room (once and
several times over), and more distinct values in one partition than it can
hold, which the full sort takes."""

import numpy as np
import pytest

import ngia2_amd as ng
import oracle_lib as orc

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = ng.Context(0)
    yield c
    c.close()


def unmix(h):
    """The signature whose mixed value is h: the inverse of the kernel's two
    odd products and two xors with a shift of itself."""
    m = 0xFFFFFFFF
    x = h.astype(np.uint64)
    x ^= (x >> np.uint64(13)) ^ (x >> np.uint64(26))
    x = (x * np.uint64(pow(0x85EBCA6B, -1, 1 << 32))) & np.uint64(m)
    x ^= x >> np.uint64(16)
    x = (x * np.uint64(pow(0x9E3779B1, -1, 1 << 32))) & np.uint64(m)
    return x.astype(np.uint32)


def signatures(n, seed):
    rng = np.random.default_rng(seed)
    return rng.integers(0, 1 << 32, size=(n, 64), dtype=np.uint64).astype(np.uint32)


@pytest.mark.parametrize("n", [1, 2, 63, 65, 2048, 2049, 4096, 4097, 8191, 8192, 8193, 16385, 33000])
def test_sizes(ctx, n):
    sig = signatures(n, n)
    rng = np.random.default_rng(n + 1)
    for b, values in enumerate((1, 2, 7, 30, 300, max(n // 90, 1), max(n // 100, 1), max(n // 2, 1))):
        sig[:, b] = sig[rng.integers(0, values, n) % n, b]
    print("partitioned bucketing", n, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("count", [95, 96, 97, 98, 2100, 2900, 4095, 4096, 4097, 9000, 20000])
def test_one_value_repeated(ctx, count):
    """One value `count` times among 21,000 records, spread or in a row."""
    n = 21000
    sig = signatures(n, count)
    rng = np.random.default_rng(count)
    for b in range(0, 64, 2):
        rows = rng.permutation(n)[:count] if b % 4 else np.arange(count) + min(b, n - count)
        sig[rows, b] = 12345 + b
    print("one value repeated", count, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("distinct", [3000, 3584, 3585, 4096, 4097, 12000])
@pytest.mark.parametrize("each", [1, 3])
def test_crowded_partition(ctx, distinct, each):
    """Values whose mixed bits all begin alike: one partition holds them all."""
    n = 40000
    sig = signatures(n, distinct)
    rng = np.random.default_rng(distinct + each)
    k = min(distinct * each, n)
    for b in (0, 9, 63):
        h = rng.choice(1 << 20, size=distinct, replace=False).astype(np.uint32) + np.uint32(b << 24)
        rows = rng.permutation(n)[:k]
        sig[rows, b] = unmix(h[np.arange(k) % distinct])
    print("crowded partition", distinct, each, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))
