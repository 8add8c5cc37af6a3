"""Group inserts below the dense form's 208 items a region, which the
persistent launch takes (odd regions wait for their even neighbours): filters
filled in many calls, from empty to loaded, with every grid size, with waits
that give up at once, from graphs and without; runs queued behind a long one, as
in test_gpu_insert_shift.py, on that launch's form of the shift path.  Every
filter has to be as if its segments had gone through bulk_insert.  Prints its
case before it touches the GPU."""
import numpy as np
import pytest
import torch

from tests import spec_model as S

pytestmark = pytest.mark.gpu

KEY_IS_HASH = 0x08
QS = [14, 16, 12, 15, 13]


def _fill(oracle, seed, load):
    """The keys of every filter, and the calls' segments of fewer than 208
    items a region (48 blocks of 64 quotients) on average."""
    keys = [oracle.splitmix64(seed + i, int(load * (1 << q))) for i, q in enumerate(QS)]
    steps = 16  # 0.9 x 3072 slots a region / 16 = 173 items
    return keys, [[k[s * k.size // steps:(s + 1) * k.size // steps] for k in keys] for s in range(steps)]


@pytest.mark.parametrize("graphs", [True, False])
@pytest.mark.parametrize("what", ["default", "wait bound 0", "1 workgroup a CU", "most workgroups"])
def test_many_sparse_calls(gpu, oracle, graphs, what):
    from cqf_amd.gqf import GQF, GQFGroup, to_device_u64, to_numpy_u64
    keys, calls = _fill(oracle, 700, 0.9)
    print(f"case sparse group calls graphs={graphs} {what}", flush=True)
    filters = [GQF(q) for q in QS]
    group = GQFGroup(filters, graphs=graphs)
    try:
        if what == "wait bound 0":
            group.set_wait_bound(0)
        elif what == "1 workgroup a CU":
            group.workgroups_per_cu = 1
        elif what == "most workgroups":
            for pc in range(16, 7, -1):
                try:
                    group.workgroups_per_cu = pc
                    break
                except ValueError:
                    pass
        for segs in calls:
            n = sum(s.size for s in segs)
            assert n < 208 * sum(f.info["nregions"] for f in filters)
            offsets = np.cumsum([0] + [s.size for s in segs]).tolist()
            dk = to_device_u64(np.concatenate(segs))
            group.bulk_insert(dk, offsets)
            torch.cuda.synchronize()
            got = to_numpy_u64(dk)
            for i, s in enumerate(segs):
                m = np.uint64((1 << (QS[i] + 8)) - 1)
                assert np.array_equal(got[offsets[i]:offsets[i + 1]], np.sort(oracle.hash_many(s, int(m)))), i
        for i, q in enumerate(QS):
            o = oracle.OracleQF(q)
            o.bulk_insert(keys[i].copy())
            assert np.array_equal(filters[i].export_image(), o.image()), i
            assert filters[i].status() == 0 and filters[i].layout_errors() == 0
            o.close()
    finally:
        group.close()
        for f in filters:
            f.close()


def test_sparse_call_replayed(gpu, oracle):
    """One shape's graph replayed with the table growing and eager work and
    synchronisations in between."""
    from cqf_amd.gqf import GQF, GQFGroup, to_device_u64
    keys, calls = _fill(oracle, 900, 0.6)
    print("case sparse group call replayed", flush=True)
    filters = [GQF(q) for q in QS]
    other = GQF(13)
    group = GQFGroup(filters, graphs=True)
    n = [min(c[i].size for c in calls) for i in range(len(QS))]
    offsets = np.cumsum([0] + n).tolist()
    buf = torch.empty(offsets[-1], dtype=torch.int64, device="cuda")
    oracles = [oracle.OracleQF(q) for q in QS]
    try:
        for r, segs in enumerate(calls[:5]):
            buf.copy_(to_device_u64(np.concatenate([s[:k] for s, k in zip(segs, n)])))
            group.bulk_insert(buf, offsets)
            other.bulk_insert(to_device_u64(segs[0][:100].copy()))
            torch.cuda.synchronize()
            for i, o in enumerate(oracles):
                o.bulk_insert(segs[i][:n[i]].copy())
                assert np.array_equal(filters[i].export_image(), o.image()), (r, i)
    finally:
        for o in oracles:
            o.close()
        group.close()
        other.close()
        for f in filters:
            f.close()


@pytest.mark.parametrize("run", [3, 70, 150])
@pytest.mark.parametrize("queued", [1, 4, 24, 25, 120])
def test_queued_runs_in_a_group(gpu, run, queued):
    from cqf_amd.gqf import GQF, GQFGroup, to_device_u64
    q = 12
    print(f"case group queued runs run={run} queued={queued}", flush=True)
    rng = np.random.default_rng(100 * run + queued)
    filters = [GQF(q), GQF(q)]
    group = GQFGroup(filters)
    ms = [{}, {}]

    def insert(hs):
        parts = [hs, np.flip(hs)]  # the same items for both, in two orders
        group.bulk_insert(to_device_u64(np.concatenate(parts)), [0, hs.size, 2 * hs.size], flags=KEY_IS_HASH)
        for m, p in zip(ms, parts):
            for h in p.tolist():
                m[h] = m.get(h, 0) + 1

    try:
        q0 = 64 * 20 + 50
        base = np.concatenate([(q0 << 8) + rng.permutation(256)[:run],
                               rng.integers(0, 1 << (q + 8), size=1 << (q - 1))]).astype(np.uint64)
        for lo in range(0, base.size, 200):
            insert(base[lo:lo + 200])
        for step in range(2):
            qs = q0 + 1 + np.arange(0, queued, 1 + step)
            insert(np.concatenate([(qs << 8) + rng.integers(0, 256, size=qs.size),
                                   rng.integers(0, 1 << (q + 8), size=100)]).astype(np.uint64))
            torch.cuda.synchronize()
            for f, m in zip(filters, ms):
                assert f.status() == 0 and f.layout_errors() == 0
                assert f.export_image().tobytes() == S.build_image(q, m)
    finally:
        group.close()
        for f in filters:
            f.close()


def test_autotune_of_a_dense_shape_leaves_the_grid(gpu, oracle):
    """A batch that takes the dense form has no grid: what sparse batches use
    stays as it was set; a sparse shape's grid is one of the candidates."""
    from cqf_amd.gqf import GQF, GQFGroup
    print("case autotune dense and sparse shapes", flush=True)
    filters = [GQF(q) for q in QS]
    group = GQFGroup(filters)
    try:
        group.workgroups_per_cu = 3
        regions = [f.info["nregions"] for f in filters]
        group.autotune(np.cumsum([0] + [1000 * r for r in regions]).tolist())
        assert group.workgroups_per_cu == 3
        group.autotune(np.cumsum([0] + [100 * f.info["nregions"] for f in filters]).tolist())
        assert group.workgroups_per_cu in (4, 6, 8, 10, 12, 16)
    finally:
        group.close()
        for f in filters:
            f.close()
