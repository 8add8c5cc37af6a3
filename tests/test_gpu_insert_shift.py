"""The insert path that moves bytes by a shift, on small tables against the
spec model's canonical image: batches of at most 208 items a region whose new
runs meet where it can go wrong: many quotients whose runs all start at one
slot (behind a long run, so one position's growth passes what a 2-bit field
holds), shifts on both sides of the 24 slots the straight pass carries, old
runs that cross one and several blocks, a full cluster up to the window's
last blocks.  Prints its case before it touches the GPU."""
import numpy as np
import pytest
import torch

from tests import spec_model as S

pytestmark = pytest.mark.gpu

KEY_IS_HASH = 0x08


@pytest.mark.parametrize("run", [3, 8, 70, 150])           # slots of the long run the others queue behind
@pytest.mark.parametrize("group", [1, 2, 3, 4, 23, 24, 25, 120])  # new quotients queued behind it
def test_queued_runs(gpu, run, group):
    from cqf_amd.gqf import GQF, to_device_u64
    print(f"case queued runs run={run} group={group}", flush=True)
    q = 12
    rng = np.random.default_rng(100 * run + group)
    ms = {}
    f = GQF(q)
    try:
        # a long run, then loose quotients over the table, half of the slots
        q0 = 64 * 20 + 50
        base = np.concatenate([(q0 << 8) + rng.permutation(256)[:run],
                               rng.integers(0, 1 << (q + 8), size=1 << (q - 1))]).astype(np.uint64)
        for lo in range(0, base.size, 400):
            part = base[lo:lo + 400]
            f.bulk_insert(to_device_u64(part), flags=KEY_IS_HASH)
            for h in part.tolist():
                ms[h] = ms.get(h, 0) + 1
        for step in range(2):  # one item for each queued quotient, then a second one for half of them
            qs = q0 + 1 + np.arange(0, group, 1 + step)
            hs = np.concatenate([(qs << 8) + rng.integers(0, 256, size=qs.size),
                                 rng.integers(0, 1 << (q + 8), size=200)]).astype(np.uint64)
            f.bulk_insert(to_device_u64(hs), flags=KEY_IS_HASH)
            for h in hs.tolist():
                ms[h] = ms.get(h, 0) + 1
            torch.cuda.synchronize()
            assert f.status() == 0 and f.layout_errors() == 0
            assert f.export_image().tobytes() == S.build_image(q, ms)
    finally:
        f.close()
