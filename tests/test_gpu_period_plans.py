"""Period scores of sizes that are planned in different ways (one pass over the
values, several, a ragged last chunk, sums from stored block sums of a pass or
straight from the values), many tensors per call, against the oracle: float64 sums
in another order, so 1e-12 relative, and against NaN, infinite and invalid inputs."""

import numpy as np
import pytest
import torch

import gpu_util as gu
from gefen_amd.partitioning import candidate_divisors, divisors
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

# powers of two up to and past a chunk, highly composite (several passes), primes times
# little (no chunk divides them), primes beyond a chunk, two large primes
SIZES = [4, 5, 9, 511, 512, 2048, 4095, 4096, 4097, 8192, 5001, 7 * 32003, 12 * 10501, 768 * 29 * 4, 55440, 720720,
         1499 * 1500, 4 * 7919, 263 * 269, 1 << 18, 3 << 17, 2 * 3 * 5 * 7 * 11 * 13, 128 * 4099, 8191 * 8]


def _values(n, dtype, seed):
    rng = np.random.default_rng(seed)
    scale = np.exp2(rng.integers(-14, -3, (n + 47) // 48)).repeat(48)[:n]
    return torch.from_numpy((rng.standard_normal(n) * scale).astype(np.float32)).to(gu.TORCH[dtype])


@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_scores_of_many_sizes_in_one_call(dtype):
    from gefen_amd.kernels.period_variance import period_scores_tasks

    items, host = [], []
    for i, n in enumerate(SIZES + SIZES[5:9]):  # some sizes twice: they share launches
        v = _values(n, dtype, i)
        buf = torch.zeros(n + 1, dtype=v.dtype, device="cuda:0")  # odd offsets: no alignment is assumed
        buf[i % 2:i % 2 + n] = v.to("cuda:0")
        items.append((buf[i % 2:i % 2 + n], candidate_divisors(n)))
        host.append(v)
    got = period_scores_tasks(items, 1, 1e-12)
    for (t, divs), v, s in zip(items, host, got):
        ref = orc.period_scores(gu.to_np(v), dtype, divs, mode=1)
        np.testing.assert_allclose(s[:-1], ref, rtol=1e-12, atol=0, err_msg=str(t.numel()))
        assert s[-1] == 0


@pytest.mark.parametrize("n,period", [(8192, 4096), (3 * 10007, 10007), (4 * 6000, 6000), (2 * 65536, 65536), (6, 3),
                                      (2 * 7919, 7919), (100, 1), (4096 * 6, 8192)])
def test_one_period_alone(n, period):
    from gefen_amd.kernels.period_variance import average_adjacent_log_block_mean_difference_cuda_kernel as f

    v = _values(n, "f32", n)
    ref = orc.period_scores(v.numpy(), "f32", [period], mode=2)[0]
    assert abs(f(v.to("cuda:0"), period, input_is_squared=False, epsilon=1e-12) - ref) <= 1e-12 * abs(ref)


@pytest.mark.parametrize("n", [4096, 3 * 10007, 768 * 29, 2 * 7919])
def test_special_values(n):
    """Extremes of the logarithm (zeros, subnormals, the largest floats), then NaN and
    infinities, which the scores carry, and negative inputs, which are counted."""
    from gefen_amd.kernels.period_variance import period_scores_tasks

    divs = [d for d in divisors(n) if n // d >= 2]
    v = torch.zeros(n)
    v[::3], v[1::7], v[2::11], v[5::13] = 1e-45, 3.4e38, 1.0, 1.0 + 2.0 ** -23
    t = v.to("cuda:0")
    for mode, eps in ((0, 1e-12), (0, 1e-310), (2, 1e-300)):
        ref = orc.period_scores(v.numpy(), "f32", divs, mode=mode, eps=eps)
        got = period_scores_tasks([(t, divs)], mode, eps)[0]
        np.testing.assert_allclose(got[:-1], ref, rtol=1e-12, atol=0)
        assert got[-1] == 0
    t[n // 2] = float("nan")
    got = period_scores_tasks([(t, divs)], 1, 1e-12)[0]
    assert all(np.isnan(got[:-1])) and got[-1] == 0
    t[n // 2] = float("inf")
    assert not any(np.isfinite(period_scores_tasks([(t, divs)], 1, 1e-12)[0][:-1]))
    t[:] = 1.0
    t[n - 1], t[0], t[n // 3] = -1.0, -2.0, -3.0
    assert period_scores_tasks([(t, divs)], 0, 1e-12)[0][-1] == 3
