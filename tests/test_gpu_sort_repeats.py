"""Sorts of batches that repeat their keys, at every form a crowded bucket can
take: one workgroup's sort by digits, a bucket in LDS, by a table of its
distinct keys (values with many copies, more of them than are listed), and
between global buffers; plain batches and sequenced ones, whose repeats differ
by their requests.  The batch is counted into a table and deleted again, so the
regions that the sort finds have to be right for the table to end up empty.
Every test prints its case before it touches the GPU."""
import numpy as np
import pytest
import torch

from tests.test_gpu_sort_sizes import _hash

pytestmark = pytest.mark.gpu


def _keys(oracle, q, kind, n, rng):
    pool = oracle.splitmix64(17, 1 << 19)
    h = _hash(pool, q + 8)
    if kind.startswith("hot"):  # that many keys, over and over
        return pool[rng.integers(0, int(kind[3:]), size=n)]
    if kind == "half":          # one key is half of the batch
        k = pool[:n].copy()
        k[rng.permutation(n)[: n // 2]] = pool[0]
        return k
    top = h >> np.uint64(q + 8 - int(kind[-1]))  # keys of one bucket
    one = pool[top == np.uint64(5 % (1 << int(kind[-1])))]
    if kind.startswith("copies"):  # 70 values of it, 4200 copies each
        return np.repeat(one[:70], n // 70)[rng.permutation(n // 70 * 70)]
    return np.concatenate([one[: 5 * n // 6], pool[: n - 5 * n // 6]])[rng.permutation(n)]


CASES = [("hot1", 65), ("hot3", 200), ("hot1", 8192), ("hot100", 5000), ("half", 8192), ("hot7", 8191),
         ("hot100", 8193), ("hot100", 12000), ("half", 16385), ("hot1", 40000), ("half", 40000),
         ("hot2000", 40000), ("copies7", 294000), ("bucket3", 30000)]


@pytest.mark.parametrize("q", [21, 27])
@pytest.mark.parametrize("kind,n", CASES)
@pytest.mark.parametrize("nreq", [0, 2, 200])
def test_repeats(gpu, oracle, q, kind, n, nreq):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    print(f"case sort repeats q={q} {kind} n={n} requests={nreq}", flush=True)
    rng = np.random.default_rng(n + q)
    keys = _keys(oracle, q, kind, n, rng)
    n = keys.size
    h = _hash(keys, q + 8)
    f = GQF(q)
    try:
        f.bulk_insert_reduce(to_device_u64(keys))
        torch.cuda.synchronize()
        assert f.stats()["nelts"] == n and f.status() == 0
        dk = to_device_u64(keys)
        if nreq == 0:
            f.bulk_delete(dk)
            want = np.sort(h)
        else:
            ends = sorted({(i + 1) * n // nreq for i in range(nreq)} - {0})
            f.mutate_seq(dk, ends, [5 * i << 1 | 1 for i in range(len(ends))])
            req = np.searchsorted(np.array(ends), np.arange(n), side="right").astype(np.uint64)
            tagged = h | (np.uint64(5) * req) << np.uint64(48) | np.uint64(1 << 63)
            want = tagged[np.argsort(h, kind="stable")]
        torch.cuda.synchronize()
        assert np.array_equal(to_numpy_u64(dk), want)
        assert f.status() == 0 and f.layout_errors() == 0
        assert f.stats() == {"nelts": 0, "ndistinct_elts": 0, "noccupied_slots": 0}
    finally:
        f.close()
