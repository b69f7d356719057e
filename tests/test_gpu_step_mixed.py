"""Tensors of every row form in one gefen_step_tasks call share a launch per dtype
pair when they are small; the results are those of each tensor stepped by itself
(its own kernel), bit for bit.  Rows past the register kernel's length against the
oracle."""

import ctypes

import numpy as np
import pytest
import torch

import gpu_util as gu
from gefen_amd import _lib
from test_gpu_step import _codebook, _run_case, _tables

pytestmark = pytest.mark.gpu

# (rows, period, magnitude block of a period-one tensor)
SHAPES = [(37, 3, 0), (7, 8, 0), (33, 24, 0), (65, 250, 0), (9, 256, 0), (5, 300, 0), (6, 511, 0), (5, 1024, 0),
          (4, 1100, 0), (3, 2500, 0), (5, 4096, 0), (4, 4097, 0), (3, 8192, 0), (3, 8203, 0), (3, 9001, 0), (2, 20480, 0), (2, 70003, 0),
          (13, 1, 1), (40, 1, 4), (1000, 1, 5), (2500, 1, 125), (2560, 1, 256), (1030, 1, 103), (720, 1, 12)]


def _build(dt, sdt, seed):
    rows, tasks = [], np.zeros(len(SHAPES), dtype=_lib.STEP_TASK)
    for i, (nrows, period, pod) in enumerate(SHAPES):
        n = nrows * period
        r = torch.Generator().manual_seed(seed + i)
        p = (torch.randn(n, generator=r) * 0.02).to(gu.TORCH[dt]).cuda()
        g = (torch.randn(n, generator=r) * 0.05).to(gu.TORCH[dt]).cuda()
        if i % 4 == 1:
            g[:period * 2] = 0
        idx = torch.randint(0, 256, (n,), generator=r, dtype=torch.uint8).cuda()
        mag = (torch.rand(n // (pod or period), generator=r) * 0.05 * (i % 5 > 0)).to(gu.TORCH[sdt]).cuda()
        vm = (torch.rand(nrows, generator=r) * 1e-3).to(gu.TORCH[sdt]).cuda()
        rows.append((p, g, idx, mag, vm))
        t = tasks[i]
        for key, v in zip(("p", "grad", "m_codebook", "m_magnitude", "vmean"), rows[-1]):
            t[key] = v.data_ptr()
        t["numel"], t["period"], t["period_one_divisor"] = n, period, pod
        t["param_dtype"], t["state_dtype"] = gu.CODE[dt], gu.CODE[sdt]
        step = 3 + i % 3  # several bias corrections: several stepsize tables
        t["beta1"], t["beta2"], t["lr"], t["eps"], t["weight_decay"] = 0.9, 0.999, 1e-3, 1e-8, 0.1 * (i % 2)
        t["bias_correction_1"], t["bias_correction_2"] = 1 - 0.9 ** step, 1 - 0.999 ** step
    return rows, tasks


@pytest.mark.parametrize("dt,sdt", [("bf16", "bf16"), ("f16", "f16"), ("f32", "f32"), ("bf16", "f32"), ("f16", "f32")])
def test_mixed_launch_matches_single_steps(dt, sdt):
    lib = _lib.load()
    tables = _tables(torch.from_numpy(_codebook()).to("cuda:0"))
    (ra, ta), (rb, tb), (rc, tc), (rd, td) = (_build(dt, sdt, 500) for _ in range(4))
    plan = ctypes.c_void_p()
    _lib.check(lib.gefen_step_plan_create(tc.ctypes.data, len(tc), tables.data_ptr(), ctypes.byref(plan)))
    for _ in range(2):
        for i in range(len(ta)):
            _lib.check(lib.gefen_step_tasks(ta[i:i + 1].ctypes.data, 1, tables.data_ptr(), gu.stream()))
        _lib.check(lib.gefen_step_tasks(tb.ctypes.data, len(tb), tables.data_ptr(), gu.stream()))
        _lib.check(lib.gefen_step_plan_run(plan, tc.ctypes.data, len(tc), gu.stream()))
        _lib.check(lib.gefen_step_tasks_noalloc(td.ctypes.data, len(td), tables.data_ptr(), gu.stream()))
    torch.cuda.synchronize()
    lib.gefen_step_plan_destroy(plan)
    for i, (a, b, c, d) in enumerate(zip(ra, rb, rc, rd)):
        for key, x, y, z, w in zip(("p", "g", "idx", "mag", "vmean"), a, b, c, d):
            for other in (y, z, w):
                assert torch.equal(x.view(torch.uint8), other.view(torch.uint8)), (SHAPES[i], key)


@pytest.mark.parametrize("dt,sdt", [("bf16", "bf16"), ("f16", "f16"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("length", [4104, 8191, 8193, 16389, 100003])
def test_long_rows_match_oracle(dt, sdt, length):
    _run_case("long_{}_{}_{}".format(dt, sdt, length), dt, sdt, length * 3, length, 0.05)
