"""The block-normalised histogram over row lengths at and beside its kernels' limits
(one element, less than a vector, a shifted last vector, the register rows' end,
rows read twice), unaligned, with rows that normalise specially, one tensor at a
time and many per call: counts equal the oracle's exactly."""

import numpy as np
import pytest
import torch

import gpu_util as gu
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

ROWS = [1, 2, 3, 4, 5, 7, 8, 9, 12, 31, 64, 65, 250, 256, 257, 511, 512, 513, 1023, 1025, 2047, 2048, 2049, 4095, 4096,
        4097, 5003]


def _values(rows, length, dtype, seed):
    rng = np.random.default_rng(seed)
    v = rng.standard_normal((rows, length)).astype(np.float32)
    v *= np.exp2(rng.integers(-12, 3, (rows, 1))).astype(np.float32)
    if dtype == "f32":
        # maxima outside the fast quotient's range, and quotients that lose bits
        for r, scale in zip(range(2, rows), (1e-30, 1e-37, 1e-42, 3e37)):
            v[r] *= np.float32(scale)
        v[-1, ::2] *= np.float32(2.0 ** -100)
    v[0] = 0.0
    if rows > 8:
        v[6, length // 2], v[7, length // 3], v[8, 0] = np.nan, np.inf, -np.inf
    return torch.from_numpy(v.reshape(-1)).to(gu.TORCH[dtype])


def _cases(dtype):
    out = []
    for i, length in enumerate(ROWS):
        rows = max(11, min(400, 40000 // length)) if length > 1 else 20011
        out.append((_values(rows, length, dtype, i), length))
    return out


def _device(v, i):
    buf = torch.zeros(v.numel() + 3, dtype=v.dtype, device="cuda:0")
    buf[i % 3:i % 3 + v.numel()] = v.to("cuda:0")  # no alignment is assumed
    return buf[i % 3:i % 3 + v.numel()]


def _ref(v, length, dtype, bins):
    counts = np.zeros(bins, dtype=np.int64)
    orc.histogram(gu.to_np(v), dtype, length, bins, counts)
    return counts


@pytest.mark.parametrize("bins", [4096, 256, 1000, 1])
@pytest.mark.parametrize("dtype", ["f32", "bf16", "f16"])
def test_counts_equal_the_oracle(dtype, bins):
    from gefen_amd.kernels.exact_histogram_fused import accumulate_histograms, gefen_exact_histogram_cuda

    cases = _cases(dtype)
    dev = [_device(v, i) for i, (v, _) in enumerate(cases)]
    want = np.zeros(bins, dtype=np.float32)
    for t, (v, length) in zip(dev, cases):
        ref = _ref(v, length, dtype, bins)
        counts = torch.full((bins,), 3, dtype=torch.int64, device="cuda:0")
        gefen_exact_histogram_cuda(t, length, counts)
        np.testing.assert_array_equal(counts.cpu().numpy() - 3, ref, err_msg=str(length))
        want = want + ref.astype(np.float32)
    acc = torch.zeros(bins, dtype=torch.float32, device="cuda:0")
    accumulate_histograms([(t, length) for t, (_, length) in zip(dev, cases)], acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), want)


def test_many_tensors_sum_in_order():
    """More tensors than one launch's table holds, with counts past 2^24 in the sum, so
    that the float32 sum depends on its order."""
    from gefen_amd.kernels.exact_histogram_fused import accumulate_histograms

    acc = torch.full((4096,), 2.0 ** 24 + 2, dtype=torch.float32, device="cuda:0")
    want = acc.cpu().numpy().copy()
    items = []
    for i in range(130):
        v = _values(12 + i, 48 + (i % 3) * 200, "f32", i)
        items.append((_device(v, 0), 48 + (i % 3) * 200))
        want = want + _ref(v, 48 + (i % 3) * 200, "f32", 4096).astype(np.float32)
    accumulate_histograms(items, acc)
    np.testing.assert_array_equal(acc.cpu().numpy(), want)


def test_counts_of_many_tensors_stay_small():
    """The tensors' own counts (32 KB each) are formed a bounded number of tensors at a time."""
    from gefen_amd.kernels.exact_histogram_fused import accumulate_histograms

    v = torch.randn(3000 * 64, generator=torch.Generator().manual_seed(5)).cuda()
    items = [(v[i * 64:(i + 1) * 64], 16) for i in range(3000)]
    acc = torch.zeros(4096, dtype=torch.float32, device="cuda:0")
    torch.cuda.synchronize()
    torch.cuda.reset_peak_memory_stats()
    before = torch.cuda.memory_allocated()
    accumulate_histograms(items, acc)
    torch.cuda.synchronize()
    assert torch.cuda.max_memory_allocated() - before <= 40 << 20
    want = np.zeros(4096, dtype=np.float32)
    for i in range(3000):
        want += _ref(v[i * 64:(i + 1) * 64], 16, "f32", 4096).astype(np.float32)
    np.testing.assert_array_equal(acc.cpu().numpy(), want)
