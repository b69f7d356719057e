"""The 256 x 256 tile of the batched Newton-Schulz products, which launches of whole
rounds of tiles take, against the one-matrix kernel, bit for bit: D by rows and
transposed, symmetric products, C together with C^T, the Gram product from X^T, and
the fused updates of every parameter dtype and orientation.  Each case asserts that
its launches take that tile."""

import math

import numpy as np
import pytest
import torch

import gpu_util as gu
import test_gpu_ns_padded as padded
from gefen_amd import _lib

pytestmark = pytest.mark.gpu


def _takes_large_tile(batch, m, n, k, symmetric):
    return _lib.load().gefen_gemm_bf16_nt_batched_tile(batch, m, n, k, int(symmetric)) == 256


def _rand(shape, seed):
    gen = torch.Generator(device="cuda:0").manual_seed(seed)
    return (torch.randn(shape, generator=gen, device="cuda:0") * 0.05).bfloat16()


def _equal(a, b):
    return torch.equal(a.contiguous().view(torch.int16), b.contiguous().view(torch.int16))


@pytest.mark.parametrize("d", ["none", "rows", "transposed"])
@pytest.mark.parametrize("outputs", ["c", "ct", "both"])
@pytest.mark.parametrize("g,m,n,k", [(52, 512, 512, 64), (104, 512, 256, 192), (26, 1024, 512, 512)])
def test_products(g, m, n, k, outputs, d):
    from gefen_amd.newton_schulz import gemm, gemm_nt_batched

    assert _takes_large_tile(g, m, n, k, False)
    a, b = _rand((g, m, k), 1), _rand((g, n, k), 2)
    dd = _rand((g, m, n), 3) if d != "none" else None
    out = torch.empty(g, m, n, dtype=torch.bfloat16, device="cuda:0") if outputs != "ct" else None
    out_t = torch.empty(g, n, m, dtype=torch.bfloat16, device="cuda:0") if outputs != "c" else None
    beta = 0.0 if dd is None else -1.25
    gemm_nt_batched(a, b, out, out_t=out_t, d=dd if d == "rows" else None,
                    d_t=dd.transpose(1, 2).contiguous() if d == "transposed" else None, alpha=0.7, beta=beta)
    want = torch.empty(g, m, n, dtype=torch.bfloat16, device="cuda:0")
    for i in range(g):
        gemm(a[i], b[i], True, want[i], d=None if dd is None else dd[i], alpha=0.7, beta=beta)
    torch.cuda.synchronize()
    assert out is None or _equal(out, want)
    assert out_t is None or _equal(out_t, want.transpose(1, 2))


@pytest.mark.parametrize("d", ["none", "rows", "transposed"])
@pytest.mark.parametrize("g,m,k", [(80, 512, 64), (40, 768, 128)])
def test_symmetric_products_and_gram(g, m, k, d):
    from gefen_amd.newton_schulz import gemm, gemm_nt_batched, gram_batched

    assert _takes_large_tile(g, m, m, k, True)
    x = _rand((g, m, k), 4)
    dd = None
    if d != "none":
        dd = _rand((g, m, m), 5)
        dd = (dd + dd.transpose(1, 2)).contiguous()
    beta = 0.0 if dd is None else -4.775
    out = torch.empty(g, m, m, dtype=torch.bfloat16, device="cuda:0")
    gemm_nt_batched(x, x, out, d=dd if d == "rows" else None, d_t=dd if d == "transposed" else None, alpha=2.0315,
                    beta=beta, symmetric=True)
    want = torch.empty_like(out)
    for i in range(g):
        gemm(x[i], x[i], True, want[i], d=None if dd is None else dd[i], alpha=2.0315, beta=beta)
    torch.cuda.synchronize()
    assert _equal(out, want)
    if dd is None:
        gram_batched(x.transpose(1, 2).contiguous(), out)
        for i in range(g):
            gemm(x[i], x[i], True, want[i])
        torch.cuda.synchronize()
        assert _equal(out, want)


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float16, torch.float32])
@pytest.mark.parametrize("batch", [52, 116])  # one launch, and one of 64 matrices (the most) with one of 52
def test_fused_update(batch, dtype, transposed):
    from gefen_amd.newton_schulz import gemm, gemm_nt_batched_apply

    m, n, k = 256, 1024, 64
    assert all(_takes_large_tile(nb, m, n, k, False) for nb in ((52,) if batch == 52 else (64, 52)))
    a, b, d_t = _rand((batch, m, k), 6), _rand((batch, n, k), 7), _rand((batch, n, m), 8)
    shape = (n, m) if transposed else (m, n)
    p = _rand((batch,) + shape, 9).to(dtype)
    want = p.clone()
    code = {torch.float32: gu.CODE["f32"], torch.float16: gu.CODE["f16"], torch.bfloat16: gu.CODE["bf16"]}[dtype]
    u = torch.empty((batch,) + shape, dtype=torch.bfloat16, device="cuda:0")
    for i in range(batch):
        one = torch.empty(m, n, dtype=torch.bfloat16, device="cuda:0")
        gemm(a[i], b[i], True, one, d=d_t[i].T.contiguous(), alpha=1.0, beta=3.4445)
        u[i] = one.T if transposed else one

    def tasks(params, update):
        t = np.zeros(batch, dtype=_lib.MUON_APPLY_TASK)
        for i in range(batch):
            t[i]["p"], t[i]["update"] = params[i].data_ptr(), update[i].data_ptr() if update is not None else 0
            t[i]["numel"], t[i]["param_dtype"], t[i]["transposed"] = m * n, code, int(transposed)
            t[i]["lr"], t[i]["weight_decay"] = 0.02, 0.1 * (i % 2)
            t[i]["adjusted_lr"] = 0.02 * 0.2 * math.sqrt(max(m, n)) * (1 + i % 3)
        return t

    gemm_nt_batched_apply(a, b, d_t, 1.0, 3.4445, tasks(p, None))
    t = tasks(want, u)
    _lib.check(_lib.load().gefen_muon_apply_tasks(t.ctypes.data, batch, gu.stream()))
    torch.cuda.synchronize()
    assert torch.equal(p.view(torch.uint8), want.view(torch.uint8))


@pytest.mark.parametrize("rows,cols,dtype,offset", [(500, 508, torch.float16, 0), (508, 500, torch.bfloat16, 1),
                                                    (500, 500, torch.float32, 0)])
def test_padded_stack(rows, cols, dtype, offset):
    """Parameters that end inside a large tile."""
    assert _takes_large_tile(64, 512, 512, 512, False)
    padded.test_padded_stack_equals_one_matrix_products(64, rows, cols, dtype, offset, 1)
