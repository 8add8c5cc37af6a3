"""The search of a sequenced query for its hash's first mutation item
(qf_bulk_get_seq_adjust), over sorted items that its guesses fit and do not
fit: spread evenly, crowded at one end or in the middle, all one hash, few
items, long stretches of one hash.  The count of a query that follows only
inserts is the number of items with its hash."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

Q = 16
TOP = (1 << (Q + 8)) - 1


def _items(kind, n, rng):
    even = rng.integers(0, TOP + 1, size=n)
    if kind == "even":
        return even
    if kind == "low":
        return even >> 12
    if kind == "high":
        return TOP - (even >> 12)
    if kind == "middle":
        return (TOP >> 1) + (even >> 14)
    if kind == "ends":
        return np.where(even & 1, even >> 16, TOP - (even >> 16))
    if kind == "one":
        return np.full(n, int(even[0]))
    assert kind == "runs"
    return np.sort(even)[(np.arange(n) // 700) * 700]


@pytest.mark.parametrize("n", [1, 2, 31, 33, 64, 5000, 200000])
@pytest.mark.parametrize("kind", ["even", "low", "high", "middle", "ends", "one", "runs"])
def test_first_item(gpu, oracle, kind, n):
    import torch
    from cqf_amd.gqf import GQF, to_device_u64
    print(f"case {kind} n={n}", flush=True)
    rng = np.random.default_rng(n)
    mut = np.sort(_items(kind, n, rng)).astype(np.uint64)
    near = rng.choice(mut, size=300)
    ask = np.concatenate([near, np.minimum(near + 1, TOP), np.maximum(near, 1) - 1, rng.integers(0, TOP + 1, size=300),
                          mut[:1], mut[-1:], [0, TOP]]).astype(np.uint64)
    keys = np.array([oracle.hash_64i(int(h), TOP) for h in ask], dtype=np.uint64)
    want = np.searchsorted(mut, ask, "right") - np.searchsorted(mut, ask, "left")
    f = GQF(Q)
    try:
        counts = torch.zeros(ask.size, dtype=torch.int64, device="cuda")
        f.get_seq_adjust(to_device_u64(keys), [ask.size], [5], counts, to_device_u64(mut))
        torch.cuda.synchronize()
        assert np.array_equal(counts.cpu().numpy(), want)
    finally:
        f.close()
