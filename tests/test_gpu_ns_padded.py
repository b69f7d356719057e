"""Newton-Schulz on zero-padded stacks with the update applied in the last product
(gefen_newton_schulz_apply), against the one-matrix products fed the same
normalised matrices and gefen_muon_apply_tasks: bit for bit (zero rows and columns
add exact zeros at the end of every K sum, and all tiles sum K in one order)."""

import numpy as np
import pytest
import torch

import gpu_util as gu

pytestmark = pytest.mark.gpu

COEFFS = (3.4445, -4.7750, 2.0315)


# sides at and beside the tiles (128, 256) and the 8-element chunks, tall and wide,
# one matrix and stacks, more matrices than one launch's table holds (64)
@pytest.mark.parametrize("batch,rows,cols,dtype,offset", [
    (3, 129, 257, torch.bfloat16, 0),
    (2, 257, 129, torch.bfloat16, 1),
    (1, 7, 300, torch.float32, 0),
    (2, 300, 7, torch.float32, 3),
    (2, 256, 384, torch.float32, 0),
    (2, 384, 256, torch.bfloat16, 0),
    (2, 200, 648, torch.float16, 0),
    (66, 130, 136, torch.bfloat16, 0),
    (40, 520, 500, torch.float32, 0),
    (1, 1, 200, torch.bfloat16, 0),
])
@pytest.mark.parametrize("steps", [1, 2])
def test_padded_stack_equals_one_matrix_products(batch, rows, cols, dtype, offset, steps):
    from gefen_amd import _lib
    from gefen_amd.newton_schulz import gemm

    lib = _lib.load()
    a, b, c = COEFFS
    gen = torch.Generator().manual_seed(batch + rows * 3 + cols * 7)
    x = (torch.randn(batch, rows, cols, generator=gen) * 1e-3).bfloat16().cuda()
    sumsq = torch.zeros(batch * 128, dtype=torch.float64, device="cuda:0")
    sumsq.view(batch, 8, 16)[:, 0, 0] = x.double().square().sum(dim=(1, 2))
    index = torch.arange(batch, dtype=torch.int32, device="cuda:0")
    n = rows * cols
    flat = (torch.randn(batch * n + 8, generator=gen) * 0.02).to(dtype).cuda()
    want = flat.clone()
    tasks = np.zeros(batch, dtype=_lib.MUON_APPLY_TASK)
    for i in range(batch):
        t = tasks[i]
        t["p"] = flat.data_ptr() + (offset + i * n) * flat.element_size()
        t["numel"], t["transposed"] = n, int(rows > cols)
        t["param_dtype"] = {torch.float32: 0, torch.float16: 1, torch.bfloat16: 2}[dtype]
        t["lr"], t["weight_decay"], t["adjusted_lr"] = 0.02, 0.1 * (i % 2), 0.02 * (1 + i % 3)
    ref_tasks = tasks.copy()
    work = torch.empty(int(lib.gefen_newton_schulz_workspace_size(batch, rows, cols)), dtype=torch.uint8,
                       device="cuda:0")
    work.fill_(0xFF)  # every padded element the products read has been written
    _lib.check(lib.gefen_newton_schulz_apply(x.data_ptr(), batch, rows, cols, a, b, c, steps, 1e-7, sumsq.data_ptr(),
                                             index.data_ptr(), work.data_ptr(), tasks.ctypes.data, gu.stream()))
    keep = []
    for i in range(batch):
        m = x[i].T.contiguous() if rows > cols else x[i].contiguous()
        norm = float(x[i].double().square().sum().sqrt().float().bfloat16())
        m = (m.float() / norm).bfloat16()
        gram = torch.empty(m.shape[0], m.shape[0], dtype=torch.bfloat16, device="cuda:0")
        upd, nxt = torch.empty_like(gram), torch.empty_like(m)
        for _ in range(steps):
            gemm(m, m, True, gram)
            gemm(gram, gram, False, upd, d=gram, alpha=c, beta=b)
            gemm(upd, m, False, nxt, d=m, alpha=1.0, beta=a)
            m, nxt = nxt, m
        u = (m.T if rows > cols else m).contiguous()
        keep.append(u)
        ref_tasks[i]["p"] = want.data_ptr() + (offset + i * n) * want.element_size()
        ref_tasks[i]["update"] = u.data_ptr()
        torch.cuda.synchronize()
    _lib.check(lib.gefen_muon_apply_tasks(ref_tasks.ctypes.data, batch, gu.stream()))
    torch.cuda.synchronize()
    assert torch.equal(flat.view(torch.uint8), want.view(torch.uint8))


def test_padded_call_refuses_what_it_cannot_take():
    from gefen_amd import _lib

    lib = _lib.load()
    assert lib.gefen_newton_schulz_workspace_size(1, 40000, 40000) == 0
    x = torch.zeros(1, 130, 140, dtype=torch.bfloat16, device="cuda:0")
    p = torch.zeros(130 * 140, device="cuda:0")
    s = torch.zeros(128, dtype=torch.float64, device="cuda:0")
    t = np.zeros(1, dtype=_lib.MUON_APPLY_TASK)
    t[0]["p"], t[0]["numel"] = p.data_ptr(), 130 * 140
    work = torch.empty(int(lib.gefen_newton_schulz_workspace_size(1, 130, 140)), dtype=torch.uint8, device="cuda:0")

    def call(rows=130, cols=140, steps=1):
        return lib.gefen_newton_schulz_apply(x.data_ptr(), 1, rows, cols, *COEFFS, steps, 1e-7, s.data_ptr(), None,
                                             work.data_ptr(), t.ctypes.data, gu.stream())

    assert call(steps=0) == 1 and call(rows=40000, cols=40000) == 1
    t[0]["transposed"] = 1
    assert call() == 1
    t[0]["transposed"], t[0]["numel"] = 0, 5
    assert call() == 1


def _low_rank_run(bound, monkeypatch):
    """Two steps of GefenMuon on 64 matrices of 8 x 14336 (29 MB; padded all at once, a
    workspace of 0.47 GB) and 3 of 30 x 9000: the parameters, and the device memory that
    the optimizer holds and held at most."""
    from gefen_amd import GefenMuon, newton_schulz

    if bound is not None:
        monkeypatch.setattr(newton_schulz, "_PADDED_WORKSPACE", bound)
        monkeypatch.setattr(newton_schulz, "_PADDED_MAX_WASTE", 0)
    gen = torch.Generator(device="cuda:0").manual_seed(4)
    shapes = [(8, 14336)] * 64 + [(30, 9000)] * 3
    ps = [torch.nn.Parameter(torch.randn(s, generator=gen, device="cuda:0") * 0.02) for s in shapes]
    for p in ps:
        p.grad = torch.randn(p.shape, generator=gen, device="cuda:0") * 1e-3
    torch.cuda.synchronize()
    before = torch.cuda.memory_allocated()
    torch.cuda.reset_peak_memory_stats()
    opt = GefenMuon([("p{}".format(i), p) for i, p in enumerate(ps)], lr=0.02)
    for _ in range(2):
        opt.step()
    torch.cuda.synchronize()
    held, peak = torch.cuda.memory_allocated() - before, torch.cuda.max_memory_allocated() - before
    return [p.detach().clone() for p in ps], held, peak


def test_padded_workspace_is_bounded():
    """Matrices that padding would grow many times over run through one bounded
    workspace, and the bound does not change a bit of the result."""
    with pytest.MonkeyPatch.context() as patch:
        want, held, peak = _low_rank_run(None, patch)
    assert peak < (256 << 20) + 6 * 30e6, (held, peak)
    with pytest.MonkeyPatch.context() as patch:
        got, held, _ = _low_rank_run(20 << 20, patch)
    assert held < (20 << 20) + 4 * 30e6, held
    for a, b in zip(want, got):
        assert torch.equal(a, b)
