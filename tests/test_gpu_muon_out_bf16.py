"""GefenMuon's momentum kernels writing the Newton-Schulz input (out_bf16) directly:
the bf16 rounding of the blend they write otherwise, bit for bit, with the same
indices and magnitudes, and the sums of squares of the bf16 values (float32 sums
per lane and workgroup, added in float64: within 1e-5 of a float64 sum)."""

import numpy as np
import pytest
import torch

import gpu_util as gu
from golden_util import load

pytestmark = pytest.mark.gpu


# (elements, block): vector rows, row tables, three vectors per lane, odd rows, one
# element per row, rows longer than a wave holds
CASES = [(4096, 256), (8192, 2048), (12 * 1536, 1536), (7 * 333, 333), (64, 1), (3 * 20001, 20001), (5 * 12, 12)]


@pytest.mark.parametrize("dtype", ["f32", "f16"])
@pytest.mark.parametrize("offset", [0, 1, 4])  # elements from an aligned address of the bf16 output
def test_bf16_output_is_the_rounded_blend(dtype, offset):
    from gefen_amd import _lib

    lib = _lib.load()
    data, _ = load("exact_dp")
    cb = torch.from_numpy(data["hist_k256_forced/codebook"]).to("cuda:0")
    tables = torch.empty(int(lib.gefen_codebook_tables_size()), dtype=torch.uint8, device="cuda:0")
    _lib.check(lib.gefen_prepare_codebook(cb.data_ptr(), cb.numel(), tables.data_ptr(), gu.stream()))
    tdt = {"f32": torch.float32, "f16": torch.float16}[dtype]
    gen = torch.Generator().manual_seed(offset + len(dtype))
    outs = {}
    grads = [(torch.randn(n, generator=gen) * 0.03).to(tdt).to("cuda:0") for n, _ in CASES]
    for half in (0, 1):
        tasks = np.zeros(len(CASES), dtype=_lib.MUON_TASK)
        keep = []
        for i, (n, block) in enumerate(CASES):
            idx = (torch.arange(n, device="cuda:0") * 37 % 256).to(torch.uint8)
            mag = torch.full((n // block,), 0.02, dtype=tdt, device="cuda:0")
            buf = torch.zeros(n + 8, dtype=torch.bfloat16 if half else tdt, device="cuda:0")
            out = buf[offset * half:offset * half + n]
            keep.append((idx, mag, out, buf))
            t = tasks[i]
            t["grad"], t["m_codebook"], t["m_magnitude"] = grads[i].data_ptr(), idx.data_ptr(), mag.data_ptr()
            t["out"], t["numel"], t["block"] = out.data_ptr(), n, block
            t["grad_dtype"] = t["state_dtype"] = gu.CODE[dtype]
            t["momentum"], t["nesterov"], t["out_bf16"] = 0.95, 1, half
        sums = torch.empty(len(CASES) * 128, dtype=torch.float64, device="cuda:0")
        _lib.check(lib.gefen_muon_tasks_sumsq(tasks.ctypes.data, len(CASES), tables.data_ptr(), sums.data_ptr(),
                                              gu.stream()))
        torch.cuda.synchronize()
        outs[half] = (keep, sums.view(len(CASES), 8, 16)[:, :, 0].sum(1))
    for i, case in enumerate(CASES):
        (idx0, mag0, out0, _), (idx1, mag1, out1, buf) = outs[0][0][i], outs[1][0][i]
        assert torch.equal(idx0, idx1) and torch.equal(mag0, mag1), case
        assert torch.equal(out0.bfloat16().view(torch.int16), out1.view(torch.int16)), case
        assert not buf[:offset].any() and not buf[offset + case[0]:].any(), case
        assert torch.allclose(outs[1][1][i], out1.double().square().sum(), rtol=1e-5, atol=0), case
