"""The step kernels on rows that are no whole number of vectors (the last vector is
shifted back over the one before it) against the oracle, with the bars of
test_gpu_step.py; and on tensors at unaligned addresses, whose rows are the aligned
ones' vectors, bit for bit against aligned copies, through gefen_step_tasks and a
kept plan."""

import ctypes

import numpy as np
import pytest
import torch

import gpu_util as gu
from gefen_amd import _lib
from gefen_amd import synthetic as syn
from oracle import oracle as orc
from test_gpu_step import _codebook, _run_case, _tables

pytestmark = pytest.mark.gpu

# one vector and a bit, lane groups' ends, whole waves with two to eight vectors per
# lane, the longest register rows and the first ones past them
LENGTHS = {"bf16": [9, 11, 15, 17, 31, 127, 250, 257, 509, 511, 515, 1021, 1027, 2047, 2049, 4090, 4095, 4097],
           "f32": [5, 6, 7, 9, 31, 127, 129, 253, 255, 257, 511, 1021, 1027, 2045, 2047, 2049]}


@pytest.mark.parametrize("dt,sdt", [("bf16", "bf16"), ("f16", "f16"), ("f32", "f32"), ("bf16", "f32"), ("f16", "f32")])
def test_odd_block_rows_match_oracle(dt, sdt):
    for i, length in enumerate(LENGTHS["f32" if dt == "f32" else "bf16"]):
        _run_case("rag_{}_{}_{}".format(dt, sdt, length), dt, sdt, length * (3 + 70 // length * (i % 2 + 1)), length,
                  0.1 * (i % 2))


@pytest.mark.parametrize("dt,sdt", [("bf16", "bf16"), ("f16", "f16"), ("f32", "f32"), ("bf16", "f32")])
@pytest.mark.parametrize("n", [9 * 1009, 251 * 67, 253 * 1013, 17 * 1021, 5 * 1013, 3 * 1019, 1021, 250 * 1009])
def test_odd_period_one_rows_match_oracle(dt, sdt, n):
    _run_case("rag_p1_{}_{}_{}".format(dt, sdt, n), dt, sdt, n, 1, 0.05)


INF = {"bf16": 0x7F80, "f16": 0x7C00, "f32": np.float32(np.inf)}
NAN = {"bf16": 0x7FC0, "f16": 0x7E00, "f32": np.float32(np.nan)}


# lane groups, whole waves of one to four vectors per lane, workgroup rows
@pytest.mark.parametrize("shared", [False, True])
@pytest.mark.parametrize("dt,sdt,length", [(dt, sdt, length) for dt, sdt in
                                           [("bf16", "bf16"), ("f16", "f16"), ("bf16", "f32"), ("f32", "f32")]
                                           for length in ([12, 250, 511, 1021, 2047, 4095] if dt != "f32" else
                                                          [6, 127, 255, 511, 1021, 2045])])
def test_infinite_gradients_in_repeated_elements(dt, sdt, length, shared):
    """Elements that the shifted last vector repeats hold +-inf, NaN and values whose
    square overflows: vmean is inf, NaN and inf, as the oracle's, in the tensor's own
    kernel and in a shared launch."""
    wide = 4 if dt == "f32" else 8
    rows = 9
    n = rows * length
    nvec = -(-length // wide)
    first, last = length - wide, (nvec - 1) * wide - 1  # the repeated elements of a row
    assert first <= last
    cb = _codebook()
    tables = _tables(torch.from_numpy(cb).to("cuda:0"))
    g = syn.round_to(syn.row_scaled_normal(5, length, rows, length, -9, -4), dt).reshape(-1).copy()
    g = g.view(np.uint16) if g.dtype == np.float16 else g
    sign = np.float32(-np.inf) if dt == "f32" else INF[dt] | 0x8000
    big = np.float32(3e38) if dt == "f32" else INF[dt] - 1  # the largest finite value
    for row, at, value in ((1, first, INF[dt]), (2, last, sign), (4, first, NAN[dt]), (6, last, big), (8, first, INF[dt])):
        g[row * length + at] = value
    p = syn.round_to(syn.normal(syn.make_key(6, length), n) * 0.02, dt)
    p = p.view(np.uint16) if p.dtype == np.float16 else p
    ref = {"p": p.copy(), "idx": np.zeros(n, np.uint8), "mag": np.zeros(rows, orc.NP_STORAGE[sdt]),
           "v": np.zeros(rows, orc.NP_STORAGE[sdt])}
    dev = {"p": gu.to_dev(p, dt), "g": gu.to_dev(g, dt), "idx": torch.zeros(n, dtype=torch.uint8, device="cuda:0"),
           "mag": torch.zeros(rows, dtype=gu.TORCH[sdt], device="cuda:0"),
           "v": torch.zeros(rows, dtype=gu.TORCH[sdt], device="cuda:0")}
    # a tensor of one-element rows asks for another kernel, so that the two share a launch
    other = {"p": torch.zeros(96, dtype=gu.TORCH[dt], device="cuda:0"), "g": torch.ones(96, dtype=gu.TORCH[dt], device="cuda:0"),
             "idx": torch.zeros(96, dtype=torch.uint8, device="cuda:0"),
             "mag": torch.zeros(32, dtype=gu.TORCH[sdt], device="cuda:0"),
             "v": torch.zeros(32, dtype=gu.TORCH[sdt], device="cuda:0")}
    tasks = np.zeros(1 + shared, dtype=_lib.STEP_TASK)
    for t, d, size, period in zip(tasks, (dev, other), (n, 96), (length, 3)):
        t["p"], t["grad"], t["m_codebook"] = d["p"].data_ptr(), d["g"].data_ptr(), d["idx"].data_ptr()
        t["m_magnitude"], t["vmean"] = d["mag"].data_ptr(), d["v"].data_ptr()
        t["numel"], t["period"] = size, period
        t["param_dtype"], t["state_dtype"] = gu.CODE[dt], gu.CODE[sdt]
        t["beta1"], t["beta2"], t["lr"], t["eps"] = 0.9, 0.999, 1e-3, 1e-8
        t["bias_correction_1"], t["bias_correction_2"] = 0.1, 1 - 0.999
    _lib.check(_lib.load().gefen_step_tasks(tasks.ctypes.data, len(tasks), tables.data_ptr(), gu.stream()))
    rc = orc.lib().orc_gefen_step(gu.CODE[dt], gu.CODE[sdt], orc._ptr(ref["p"]), orc._ptr(np.ascontiguousarray(g)),
                                  orc._ptr(ref["idx"]), orc._ptr(ref["mag"]), orc._ptr(ref["v"]), n, length, 0,
                                  orc._ptr(cb), cb.size, 0.9, 0.999, 1e-3, 1e-8, 0.0, 0.1, 1 - 0.999, 1)
    assert rc == 0
    torch.cuda.synchronize()
    np.testing.assert_array_equal(gu.to_np(dev["idx"]), ref["idx"])
    np.testing.assert_array_equal(orc.to_f32(gu.to_np(dev["mag"]), sdt), orc.to_f32(ref["mag"], sdt))
    v, w = orc.to_f32(gu.to_np(dev["v"]), sdt), orc.to_f32(ref["v"], sdt)
    assert np.isinf(w[[1, 2, 8]]).all() and np.isnan(w[4]), w
    np.testing.assert_array_equal(np.isnan(v), np.isnan(w))
    np.testing.assert_array_equal(np.isinf(v), np.isinf(w))
    np.testing.assert_array_equal(np.isnan(orc.to_f32(gu.to_np(dev["p"]), dt)), np.isnan(orc.to_f32(ref["p"], dt)))


@pytest.mark.parametrize("dt", ["bf16", "f16", "f32"])
def test_unaligned_tensors_step_as_aligned_ones(dt):
    lib = _lib.load()
    cb = torch.from_numpy(_codebook()).to("cuda:0")
    tables = _tables(cb)
    gen = torch.Generator().manual_seed(11)
    tdt = gu.TORCH[dt]
    shapes = [(40, 2048, 0), (50, 512, 0), (60, 64, 0), (256 * 40, 1, 256), (1000, 1, 250), (30, 12, 0), (9, 20, 0)]

    def build(offset):
        rows = []
        for i, (rows_v, period, pod) in enumerate(shapes):
            n = rows_v * period
            blocks = n // (pod or period)

            def at(values, dtype, shift):
                buf = torch.zeros(values.numel() + 16, dtype=dtype, device="cuda:0")
                v = buf[shift:shift + values.numel()]
                v.copy_(values)
                return v, buf

            r = torch.Generator().manual_seed(100 + i)
            p, g = torch.randn(n, generator=r) * 0.02, torch.randn(n, generator=r) * 0.05
            idx = torch.randint(0, 256, (n,), generator=r, dtype=torch.uint8)
            mag = torch.rand(blocks, generator=r) * 0.05 + 0.01
            vm = torch.rand(rows_v, generator=r) * 1e-3
            o = offset and 1 + i % 3
            rows.append([at(p, tdt, o), at(g, tdt, o), at(idx, torch.uint8, offset and 1 + i % 5), at(mag, tdt, 0),
                         at(vm, tdt, o if pod else 0)])
        tasks = np.zeros(len(shapes), dtype=_lib.STEP_TASK)
        for t, (rows_v, period, pod), r in zip(tasks, shapes, rows):
            for key, (v, _) in zip(("p", "grad", "m_codebook", "m_magnitude", "vmean"), r):
                t[key] = v.data_ptr()
            t["numel"], t["period"], t["period_one_divisor"] = rows_v * period, period, pod
            t["param_dtype"] = t["state_dtype"] = gu.CODE[dt]
            t["beta1"], t["beta2"], t["lr"], t["eps"], t["weight_decay"] = 0.9, 0.999, 1e-3, 1e-8, 0.1
            t["bias_correction_1"], t["bias_correction_2"] = 1 - 0.9 ** 3, 1 - 0.999 ** 3
        return rows, tasks

    # aligned and shifted tensors one per call (their own kernels), and the shifted ones
    # together, in a shared launch and in a plan of it
    (ra, ta), (rb, tb), (rc, tc), (rd, td) = build(0), build(1), build(1), build(1)
    out = np.zeros(1, dtype=_lib.STEP_SUMMARY)
    for tasks, shared in [(t[i:i + 1], 0) for t in (ta, tb) for i in range(len(t))] + [(tc, 1)]:
        _lib.check(lib.gefen_step_tasks_summary(tasks.ctypes.data, len(tasks), out.ctypes.data))
        assert (out[0]["launches"], out[0]["shared"]) == (1, shared)
    plan = ctypes.c_void_p()
    _lib.check(lib.gefen_step_plan_create(tc.ctypes.data, len(tc), tables.data_ptr(), ctypes.byref(plan)))
    for _ in range(2):
        for t in (ta, tb):
            for i in range(len(t)):
                _lib.check(lib.gefen_step_tasks(t[i:i + 1].ctypes.data, 1, tables.data_ptr(), gu.stream()))
        _lib.check(lib.gefen_step_plan_run(plan, tc.ctypes.data, len(tc), gu.stream()))
        _lib.check(lib.gefen_step_tasks(td.ctypes.data, len(td), tables.data_ptr(), gu.stream()))
    torch.cuda.synchronize()
    lib.gefen_step_plan_destroy(plan)
    for i, (a, b, c, d) in enumerate(zip(ra, rb, rc, rd)):
        for key, x, y, z, w in zip(("p", "g", "idx", "mag", "vmean"), a, b, c, d):
            assert torch.equal(x[0].view(torch.uint8), y[0].contiguous().view(torch.uint8)), (shapes[i], key)
            assert torch.equal(x[0].view(torch.uint8), z[0].contiguous().view(torch.uint8)), (shapes[i], key)
            assert torch.equal(x[0].view(torch.uint8), w[0].contiguous().view(torch.uint8)), (shapes[i], key)
            shift = y[0].storage_offset()
            assert not y[1][:shift].any() and not y[1][shift + y[0].numel():].any(), (shapes[i], key)  # nothing beside it
