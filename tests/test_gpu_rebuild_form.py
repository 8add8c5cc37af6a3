"""Batches near the lines between the two forms of the rebuild, with the form
found on the device: counted batches whose distinct keys (known there only) are
few or many, inserts into large tables that are empty, hardly and half loaded.
One call has to leave the table that the same keys leave in calls far below the
line.  Prints its case before it touches the GPU."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("q,per", [(9, 3), (14, 1), (14, 400), (21, 2), (22, 41), (22, 43), (22, 200)])  # keys a region
@pytest.mark.parametrize("share", [1.0, 0.5, 0.02])     # of them distinct
@pytest.mark.parametrize("load", [0.0, 0.5])
def test_counted_batches(gpu, oracle, q, per, share, load):
    from cqf_amd.gqf import GQF, to_device_u64, to_numpy_u64
    print(f"case counted q={q} per={per} share={share} load={load}", flush=True)
    rng = np.random.default_rng(q * per)
    f = GQF(q)
    o = oracle.OracleQF(q)
    try:
        n = per * f.info["nregions"]
        pool = oracle.splitmix64(3 + q, max(1, int(share * n)))
        keys = np.concatenate([pool, pool[rng.integers(0, pool.size, size=n)]])[:n]
        for k, call, ref in ((oracle.splitmix64(11, int(load * (1 << q))), f.bulk_insert, o.bulk_insert),
                             (keys, f.bulk_insert_reduce, o.bulk_insert)):
            if k.size:
                dk = to_device_u64(k)
                call(dk)
                sorted_k = k.copy()
                ref(sorted_k)
                torch.cuda.synchronize()
                assert np.array_equal(to_numpy_u64(dk), sorted_k)
        assert f.status() == 0 and f.layout_errors() == 0
        assert np.array_equal(f.export_image(), o.image())
    finally:
        f.close()
        o.close()


@pytest.mark.parametrize("load", [0.0, 0.1, 0.5])
@pytest.mark.parametrize("per", [259, 300, 421])
def test_inserts_into_a_large_table(gpu, load, per):
    from cqf_amd import workloads as W
    from cqf_amd.gqf import GQF
    q = 25
    print(f"case large inserts q={q} load={load} per={per}", flush=True)
    base = W.splitmix64(1, int(load * (1 << q)), device="cuda")
    a, b = GQF(q), GQF(q)
    try:
        new = W.splitmix64(2, per * a.info["nregions"], device="cuda")
        for f in (a, b):
            for part in base.clone().split(1 << 21):
                f.bulk_insert(part)
        a.bulk_insert(new.clone())
        for part in new.clone().split(1 << 20):
            b.bulk_insert(part)
        torch.cuda.synchronize()
        assert a.status() == 0 and a.layout_errors() == 0
        assert torch.equal(a.export_image_device(), b.export_image_device())
    finally:
        a.close()
        b.close()
