"""The workgroup-wide rebuild of dense batches and the delete path, on small
tables against the spec model's canonical image of the multiset: batches on
both sides of the density where a table changes path, counters of one to
several slots (counts from 1 past 4095, more big ones in a window than its
table of them holds), runs that cross blocks, deletes that empty runs, that
rewrite counters in place without moving a byte, and that take a run's last
byte out of the next block.  Every test prints its case before it touches
the GPU."""
import numpy as np
import pytest
import torch

from tests import spec_model as S

pytestmark = pytest.mark.gpu

KEY_IS_HASH = 0x08
NO_SPACE = 0x1


def _say(*a):
    print(*a, flush=True)


def _apply(ms, hs, d):
    for h in hs.tolist():
        c = max(0, ms.get(h, 0) + d)
        if c:
            ms[h] = c
        else:
            ms.pop(h, None)


def _check(f, q, ms):
    torch.cuda.synchronize()
    assert f.status() == 0 and f.layout_errors() == 0
    assert f.export_image().tobytes() == S.build_image(q, ms)


def _hashes(rng, q, n, distinct):
    """n hashes over about `distinct` values, spread over the whole range."""
    univ = np.unique(rng.integers(0, 1 << (q + 8), size=distinct, dtype=np.uint64))
    return univ[rng.integers(0, univ.size, size=n)]


# 74 blocks at q = 12: two regions, so 416 items are the densest batch of the
# sparse path's side; 17 blocks at q = 10: one region
@pytest.mark.parametrize("q,n,distinct", [(10, 207, 207), (10, 208, 208), (10, 900, 300), (12, 415, 415),
                                          (12, 416, 416), (12, 3600, 3000), (12, 60000, 700), (14, 14000, 13000)])
@pytest.mark.parametrize("how", ["insert", "reduce", "requests"])
def test_dense_batches(gpu, oracle, q, n, distinct, how):
    from cqf_amd.gqf import GQF, to_device_u64
    _say(f"case dense q={q} n={n} distinct={distinct} {how}")
    rng = np.random.default_rng(1000 * q + n)
    f = GQF(q)
    ms = {}
    try:
        for step in range(3):  # into the empty table, then over what is there
            hs = _hashes(rng, q, n >> step, distinct >> step)
            if how == "requests":
                keys = np.array([oracle.hash_64i(int(h), (1 << (q + 8)) - 1) for h in hs], dtype=np.uint64)
                a = hs.size // 3
                f.mutate_seq(to_device_u64(keys), [a, a + a // 2, hs.size], [0, 3, 4])  # insert, delete, insert
                _apply(ms, hs[:a], 1)
                _apply(ms, hs[a:a + a // 2], -1)
                _apply(ms, hs[a + a // 2:], 1)
            else:
                (f.bulk_insert if how == "insert" else f.bulk_insert_reduce)(to_device_u64(hs), flags=KEY_IS_HASH)
                _apply(ms, hs, 1)
            try:
                S.build_image(q, ms)
            except ValueError:  # the table is full now, which the filter has to say
                torch.cuda.synchronize()
                assert f.status() & NO_SPACE
                break
            _check(f, q, ms)
    finally:
        f.close()


@pytest.mark.parametrize("nbig", [3, 64, 90])
def test_dense_big_counts(gpu, nbig):
    """Counts on both sides of 4095, `nbig` of them at least that in one
    window, raised again by a second batch."""
    from cqf_amd.gqf import GQF, to_device_u64
    q = 11
    _say(f"case big counts {nbig}")
    rng = np.random.default_rng(nbig)
    univ = rng.permutation(1 << (q + 8))[:400].astype(np.uint64)
    counts = np.concatenate([np.full(nbig, 4095), [4094, 4093, 3, 4, 257, 258, 259],
                             rng.integers(1, 4, size=393 - nbig)]).astype(np.int64)
    counts[:nbig] += rng.integers(0, 3, size=nbig)
    f = GQF(q)
    ms = {}
    try:
        for part in (np.repeat(univ, counts), np.repeat(univ[::2], 2), univ):
            f.bulk_insert(to_device_u64(rng.permutation(part)), flags=KEY_IS_HASH)
            _apply(ms, part, 1)
            _check(f, q, ms)
    finally:
        f.close()


@pytest.mark.parametrize("q,load,repeat", [(9, 0.9, 0.0), (10, 0.6, 0.5), (12, 0.9, 0.0), (12, 0.85, 0.2), (13, 0.5, 0.9)])
def test_delete_batches(gpu, q, load, repeat):
    """Deletes of one key, a few, a third with repeats and absent keys, then
    the rest."""
    from cqf_amd.gqf import GQF, to_device_u64
    _say(f"case delete q={q} load={load} repeat={repeat}")
    rng = np.random.default_rng(int(100 * load) + q)
    n = int(load * (1 << q))
    univ = rng.permutation(1 << (q + 8))[:max(1, int(n * (1 - repeat) * (0.6 if repeat else 1)))].astype(np.uint64)
    hs = np.concatenate([univ, univ[rng.integers(0, univ.size, size=max(0, int(0.5 * n * repeat)))]])
    f = GQF(q)
    ms = {}
    try:
        f.bulk_insert(to_device_u64(hs), flags=KEY_IS_HASH)
        _apply(ms, hs, 1)
        _check(f, q, ms)
        left = rng.permutation(hs)
        for k in (1, 7, 100, left.size // 3, left.size):
            batch, left = left[:k], left[k:]
            absent = rng.integers(0, 1 << (q + 8), size=k // 4, dtype=np.uint64)
            batch = rng.permutation(np.concatenate([batch, absent]))
            f.bulk_delete(to_device_u64(batch), flags=KEY_IS_HASH)
            _apply(ms, batch, -1)
            _check(f, q, ms)
    finally:
        f.close()


@pytest.mark.parametrize("home", [0, 60, 63, 64, 3071, 3072])
def test_delete_single_places(gpu, home):
    """One change at a time around a block's and a region's end: a count
    lowered in place (300 -> 299), a two-slot counter halved, a run's last
    byte removed from the next block, a run emptied in front of pushed ones."""
    from cqf_amd.gqf import GQF, to_device_u64
    q = 12
    _say(f"case delete places {home}")
    hs = [(home << 8) | 5] * 300 + [(home << 8) | r for r in (9, 9, 40)]
    hs += [((home + k) << 8) | r for k in range(1, 7) for r in (1, 200, 255)]
    hs = np.array(hs, dtype=np.uint64)
    f = GQF(q)
    ms = {}
    try:
        f.bulk_insert(to_device_u64(hs), flags=KEY_IS_HASH)
        _apply(ms, hs, 1)
        _check(f, q, ms)
        for gone in ([(home << 8) | 5], [(home << 8) | 9], [((home + 1) << 8) | 255], [((home + 6) << 8) | 255],
                     [((home + 2) << 8) | r for r in (1, 200, 255)], [(home << 8) | 5] * 299 + [(home << 8) | 7]):
            g = np.array(gone, dtype=np.uint64)
            f.bulk_delete(to_device_u64(g), flags=KEY_IS_HASH)
            _apply(ms, g, -1)
            _check(f, q, ms)
    finally:
        f.close()
