"""gefen_automatic_vmean_update on rows of no whole number of vectors, at unaligned
addresses and across the lane groups' sizes, against float64."""

import numpy as np
import pytest
import torch

import gpu_util as gu
from gefen_amd import _lib

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("gdt,sdt", [("bf16", "bf16"), ("f16", "f16"), ("f32", "f32"), ("bf16", "f32"), ("f32", "bf16")])
@pytest.mark.parametrize("period", [1, 3, 4, 7, 8, 9, 15, 17, 63, 64, 65, 250, 511, 512, 513, 2047, 2050, 4099])
def test_vmean_rows_match_float64(gdt, sdt, period):
    lib = _lib.load()
    rows = 5 + 300 // period
    gen = torch.Generator().manual_seed(period)
    for shift in (0, 1, 3):
        buf = torch.zeros(rows * period + 8)
        buf[shift:shift + rows * period] = torch.randn(rows * period, generator=gen) * 0.1
        buf = buf.to(gu.TORCH[gdt]).cuda()
        g = buf[shift:shift + rows * period]
        vm = (torch.rand(rows, generator=gen) * 1e-2).to(gu.TORCH[sdt]).cuda()
        old = vm.double().cpu().numpy()
        _lib.check(lib.gefen_automatic_vmean_update(vm.data_ptr(), gu.CODE[sdt], g.data_ptr(), gu.CODE[gdt], rows,
                                                    period, 0.75, gu.stream()))
        ms = (g.double().cpu().numpy().reshape(rows, period) ** 2).mean(1)
        want = 0.75 * old + 0.25 * ms
        # float32: each lane's chain (a vector in every 64, its tail, the butterfly), the
        # mean's division, the product with the old value and the fma; then the state's rounding
        chain = 8 * -(-period // 256) + 8 + 6 + 4
        unit, least = {"f32": (2.0 ** -24, 0.0), "bf16": (2.0 ** -8, 0.0), "f16": (2.0 ** -11, 2.0 ** -25)}[sdt]
        bar = want * (chain * 2.0 ** -24 + unit) + least
        assert np.all(np.abs(vm.double().cpu().numpy() - want) <= bar), (period, shift)
