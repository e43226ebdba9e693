"""The partitioned bucketing at its edges, against the oracle's stable sort:
record counts at the partition counts' steps and at the tiles of the scatter,
signatures repeated past a chain's length, past a partition's room (once and
several times over), and more distinct values in one partition than it can
hold, which the full sort takes."""

import os

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


@pytest.fixture(scope="module")
def small():
    os.environ["NGIA_BUCKET_SMALL"] = "1"
    try:
        c = ng.Context(0)
    finally:
        del os.environ["NGIA_BUCKET_SMALL"]
    yield c
    c.close()


@pytest.fixture(scope="module")
def few():
    os.environ["NGIA_BUCKET_FEW"] = "1"
    try:
        c = ng.Context(0)
    finally:
        del os.environ["NGIA_BUCKET_FEW"]
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


@pytest.mark.parametrize("n", [1, 2048, 2049, 8191, 8192, 8193, 8448, 12287, 12288, 12289, 16383, 16384])
def test_small(small, n):
    """At most 16,384 records: each block shape's ends; by wavefronts, the
    column's tiles of 256 and 4,096, values repeated in one round and over many."""
    sig = signatures(n, n + 7)
    rng = np.random.default_rng(n + 8)
    for b, values in enumerate((1, 2, 7, 30, 300, max(n // 3, 1))):
        sig[:, b] = sig[rng.integers(0, values, n) % n, b]
    sig[:, 8] = sig[np.arange(n) // 2, 8]  # pairs side by side
    sig[:, 9] = sig[np.arange(n) % ((n + 1) // 2), 9]  # pairs half a column apart
    sig[:, 10] = unmix(np.full(n, 0xFFFFFFFF, dtype=np.uint32))
    sig[:, 11] = unmix(np.zeros(n, dtype=np.uint32))
    print("small bucketing", n, flush=True)
    np.testing.assert_array_equal(small.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("distinct", [959, 960, 961, 1023, 1024, 1025, 3000])
def test_small_crowded_partition(small, distinct):
    """As many values in one wavefront's table as it has slots, and more."""
    n = 9000
    sig = signatures(n, distinct)
    rng = np.random.default_rng(distinct)
    for b in (0, 9, 63):
        h = rng.choice(1 << 20, size=distinct, replace=False).astype(np.uint32) + np.uint32(b << 24)
        rows = rng.permutation(n)[: min(2 * distinct, n)]
        sig[rows, b] = unmix(h[np.arange(len(rows)) % distinct])
    print("small bucketing, crowded partition", distinct, flush=True)
    np.testing.assert_array_equal(small.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("n", [1, 64, 65, 1023, 1024, 1025, 8191, 8192, 8193, 9216, 16385, 139264, 139265])
def test_few_values(few, n):
    """The tables of few values: tiles of 8,192, wavefronts of 1,024, rows of
    64 and, past 16 tiles, the prefix's second round."""
    rng = np.random.default_rng(n)
    values = np.array([1, 2, 3, 30, 400, 1000] * 11)[:64]
    sig = np.empty((n, 64), dtype=np.uint32)
    for b in range(64):
        pool = rng.integers(0, 1 << 32, size=values[b], dtype=np.uint64).astype(np.uint32)
        pool[0] = unmix(np.array([0xFFFFFFFF if b % 2 else 0], dtype=np.uint32))[0]
        sig[:, b] = pool[(rng.random(n) ** 2 * values[b]).astype(np.int64)]
    sig[:, 7] = sig[np.arange(n) // 3, 7]
    print("few values", n, flush=True)
    np.testing.assert_array_equal(few.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("values", [1400, 1700, 2046, 2047, 2048, 3000, 20000])
def test_too_many_values(few, values):
    """More values than a table takes, in one band or over its tiles."""
    n = 30000
    rng = np.random.default_rng(values)
    sig = rng.integers(0, 300, size=(n, 64)).astype(np.uint32)
    sig[:, 40] = rng.integers(0, values, n)
    sig[:, 63] = np.arange(n) // (n // values + 1)  # few in a tile
    print("too many values", values, flush=True)
    np.testing.assert_array_equal(few.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("n", [8193, 12001, 16384])
def test_small_frequent_values(small, n):
    """Values frequent enough for registers: one throughout, one in every other
    record, several in turns of different lengths that meet in a partition (16 or 32
    of them for 64 bands of six values), and one that comes back."""
    rng = np.random.default_rng(n)
    at = np.arange(n)
    print("frequent values", n, flush=True)
    for which in (np.zeros(n, np.int64), np.where(at % 2, 0, -1), at // 17 % 6, at // 64 % 6, at // 1000 % 6,
                  rng.integers(0, 6, n), np.where(rng.random(n) < 0.8, rng.integers(0, 6, n), -1),
                  np.where(at // 2048 % 2, 0, rng.integers(-1, 3, n))):
        sig = rng.integers(0, 1 << 32, size=(n, 64), dtype=np.uint64).astype(np.uint32)
        values = rng.integers(0, 1 << 32, size=(6, 64), dtype=np.uint64).astype(np.uint32)
        sig[which >= 0] = values[which[which >= 0]]
        np.testing.assert_array_equal(small.bucket(sig), orc.bucket(sig))


def families(rng, n, size, order):
    """Records of n / size signature sets: in random order, one set after another, or
    so with one of each set's records far from the others."""
    fam = rng.integers(0, max(n // size, 1), n)
    if order != "mixed":
        fam.sort()
    if order == "strays":
        stray = rng.integers(0, n, n // size)
        fam[stray] = rng.integers(0, max(n // size, 1), len(stray))
    pool = rng.integers(0, 1 << 32, size=(max(n // size, 1), 64), dtype=np.uint64).astype(np.uint32)
    return pool[fam]


@pytest.mark.parametrize("order", ["mixed", "sorted", "strays"])
@pytest.mark.parametrize("n,size", [(20000, 70), (20000, 200), (20000, 1000), (40000, 4000), (50000, 1000),
                                    (120001, 1500)])
def test_families(ctx, n, size, order):
    """Partitions of few values and long runs, within their room and past it."""
    sig = families(np.random.default_rng(n + size), n, size, order)
    print("families", n, size, order, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("distinct", [1, 2, 63, 64, 65, 200, 2000])
@pytest.mark.parametrize("size", [97, 1024, 1025, 2048, 2049, 4095, 4096, 4097, 9000])
def test_long_chains(ctx, distinct, size):
    """`size` elements in a few partitions, half of them of one value, the others of
    `distinct`: the ends of each capacity and of the values that a partition's table
    takes."""
    n = 17000
    rng = np.random.default_rng(distinct * 10000 + size)
    sig = signatures(n, size)
    for b in (0, 9, 33, 63):
        # the partition of all ones, which other records' mixed values rarely reach
        top = np.uint32(0xFFF00000)
        h = top | rng.choice(1 << 20, size=distinct + 1, replace=False).astype(np.uint32)
        rows = rng.permutation(n)[:size] if b != 33 else np.arange(size)
        which = np.where(rng.random(size) < 0.5, 0, 1 + rng.integers(0, distinct, size))
        sig[rows, b] = unmix(h[which])
    print("long chains", distinct, size, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))


@pytest.mark.parametrize("n", [20000, 50000, 300000])
@pytest.mark.parametrize("share", [0.02, 0.3, 1.0])
def test_one_frequent_value(ctx, n, share):
    """One signature set in a share of the records: partitions past their room by the
    column's scan, or the full sort instead."""
    rng = np.random.default_rng(n)
    sig = signatures(n, n + 3)
    sig[rng.random(n) < share] = sig[7]
    print("one frequent value", n, share, flush=True)
    np.testing.assert_array_equal(ctx.bucket(sig), orc.bucket(sig))
