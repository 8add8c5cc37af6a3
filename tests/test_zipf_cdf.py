"""The CDF of the Zipf workload: as near to the exact one as float64 allows,
and the same bits wherever it is formed, so that two processes draw the same
keys from a seed (a float64 scan on the GPU gave another CDF on each call, and
some of 2^26 draws went to a neighbouring id)."""
import math

import pytest
import torch

from cqf_amd import workloads as W


@pytest.mark.parametrize("n_ids", [1, 2, 1000, (1 << 16) + 1, 1 << 20])
@pytest.mark.parametrize("s", [0.0, 0.7, 1.0, 1.5, 3.0])
def test_cdf_is_exact_to_rounding(n_ids, s):
    c = W.zipf_cdf(n_ids, s)
    w = torch.arange(1, n_ids + 1, dtype=torch.float64).pow(-s).tolist()
    total = math.fsum(w)
    for k in {1, 2, n_ids // 1000, n_ids // 7, n_ids // 2, n_ids - 1} - {0}:
        if k <= n_ids:
            exact = math.fsum(w[:k]) / total
            # each side rounds two sums and their quotient
            assert abs(float(c[k - 1]) - exact) <= 6 * 2.0 ** -53 * exact, k
    assert float(c[-1]) == 1.0 and bool((c[1:] >= c[:-1]).all())


def test_cdf_sums_without_an_order():
    """The parts that are summed are whole numbers: any order of adding them
    gives the CDF's bits."""
    n_ids, s = 1 << 14, 1.5
    c = W.zipf_cdf(n_ids, s)
    w = torch.arange(1, n_ids + 1, dtype=torch.float64).pow(-s)
    scaled = (w * 2.0 ** (52 - n_ids.bit_length() - math.frexp(float(w[0]))[1])).tolist()
    unit = 2.0 ** (62 - n_ids.bit_length())
    whole, low = [int(x) for x in scaled], [round((x - int(x)) * unit) for x in scaled]
    for k in (1, 2, 77, n_ids // 2, n_ids):
        got = (float(sum(reversed(whole[:k]))) + sum(reversed(low[:k])) / unit) / (
            float(sum(whole)) + sum(low) / unit)
        assert got == float(c[k - 1]), k


@pytest.mark.gpu
@pytest.mark.parametrize("n_ids,s", [(1 << 23, 1.5), (100003, 1.1)])
def test_gpu_draws_equal_the_cpus(gpu, n_ids, s):
    print(f"case zipf draws n_ids={n_ids} s={s}", flush=True)
    want = W.zipf_cdf(n_ids, s)
    for _ in range(3):
        assert torch.equal(W.zipf_cdf(n_ids, s, "cuda").cpu(), want)
    n = 1 << 24
    cpu = W.zipf_workload(n_ids, n, s=s, seed=3)
    dev = W.zipf_workload(n_ids, n, s=s, seed=3, device="cuda")
    for a, b in zip(cpu, dev):
        assert torch.equal(a, b.cpu())
