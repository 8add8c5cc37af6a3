"""A workspace that the device has no memory for: the call says so and launches
nothing, and the filter goes on working (its workspace was taken for allocated
before, and the next batch ran on null pointers)."""
import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def test_reserve_past_the_memory(gpu, oracle):
    from cqf_amd import gqf
    print("case reserve 2^46 keys", flush=True)
    q = 14
    f = gqf.GQF(q)
    o = oracle.OracleQF(q)
    try:
        gqf.last_error()
        assert f.reserve(1 << 46) == -2
        assert gqf.last_error() != 0
        keys = oracle.splitmix64(4, 9000)
        f.bulk_insert(gqf.to_device_u64(keys))
        assert f.bulk_insert_noalloc(gqf.to_device_u64(keys[:100])) == 0
        torch.cuda.synchronize()
        o.bulk_insert(np.concatenate([keys, keys[:100]]))
        assert f.status() == 0 and gqf.last_error() == 0
        assert np.array_equal(f.export_image(), o.image())
        assert f.reserve(1 << 20) == 0
    finally:
        f.close()
        o.close()
