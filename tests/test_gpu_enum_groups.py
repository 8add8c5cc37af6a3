"""Enumeration, statistics and merges where an enumeration's groups of 62
blocks end, and where a group does not fit its window: runs that reach past
the two blocks behind the group, more large counts than its table holds.  The
expected items are the multiset the table was filled with.  Every test prints
its case before it touches the GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

KEY_IS_HASH = 0x08
EDGE = 62 * 64  # first quotient of the second group


def _fill(q, ms):
    from cqf_amd.gqf import GQF, to_device_u64
    f = GQF(q)
    hs = np.array(sorted(ms), dtype=np.uint64)
    f.bulk_insert(to_device_u64(np.repeat(hs, [ms[int(h)] for h in hs])), flags=KEY_IS_HASH)
    torch.cuda.synchronize()
    assert f.status() == 0 and f.layout_errors() == 0
    return f


def _multiset(kind):
    rng = np.random.default_rng(5)
    ms = {int(h): 1 for h in rng.integers(0, 1 << 21, size=5000)}
    if kind == "edge runs":
        for k in range(-3, 4):
            for r in range(0, 256, 1 if k == -1 else 9):
                ms[((EDGE + k) << 8) | r] = 1 + r % 3
    elif kind == "long spill":  # 600 slots from the first group's last quotients, over the whole next block
        for k in (1, 2, 3):
            for r in range(256):
                ms[((EDGE - k) << 8) | r] = 1
    elif kind == "big counts":
        for r in range(90):
            ms[(700 << 8) | r] = 4094 + r
    elif kind == "whole group pushed":  # a run of a thousand slots behind the edge
        for k in range(4):
            for r in range(256):
                ms[((EDGE + k) << 8) | r] = 1 + (r == 7) * 300
    return ms


@pytest.mark.parametrize("kind", ["plain", "edge runs", "long spill", "big counts", "whole group pushed"])
def test_enumerate_groups(gpu, kind):
    from cqf_amd.gqf import GQF, to_numpy_u64
    q = 13
    print(f"case enumeration groups: {kind}", flush=True)
    ms = _multiset(kind)
    f = _fill(q, ms)
    want = np.array(sorted(ms), dtype=np.uint64)
    cnt = np.array([ms[int(h)] for h in want], dtype=np.uint64)
    try:
        h, c = f.enumerate()
        assert np.array_equal(to_numpy_u64(h), want) and np.array_equal(to_numpy_u64(c), cnt)
        st = f.stats()
        assert st["nelts"] == int(cnt.sum()) and st["ndistinct_elts"] == want.size
        for lo, hi in ((0, 1), (EDGE - 2, EDGE), (EDGE - 1, EDGE + 1), (EDGE, EDGE + 3), (5, EDGE - 1), (EDGE + 1, 1 << q),
                       (0, EDGE), (63, 64), (64, 65)):
            h, c = f.enumerate(lo, hi)
            m = (want >> np.uint64(8) >= lo) & (want >> np.uint64(8) < hi)
            assert np.array_equal(to_numpy_u64(h), want[m]) and np.array_equal(to_numpy_u64(c), cnt[m]), (lo, hi)
        g = GQF(q)
        assert g.merge_from(f) == want.size
        assert g.status() == 0 and g.layout_errors() == 0
        assert np.array_equal(g.export_image(), f.export_image())
        g.close()
    finally:
        f.close()
