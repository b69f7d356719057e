"""The 128 x 128 tile of the batched Newton-Schulz products, which launches with few
tiles take: bit-identical to the one-matrix kernel (one K order)."""

import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("g,m,n,k", [(1, 256, 512, 256), (2, 512, 256, 64), (1, 768, 768, 192)])
def test_small_tile_products_equal_the_one_matrix_kernel(g, m, n, k):
    """Few tiles: the plain products run on 128 x 128 tiles (bit-identical)."""
    from gefen_amd.newton_schulz import gemm, gemm_nt_batched, gram_batched

    gen = torch.Generator().manual_seed(m + n + k)
    a = (torch.randn(g, m, k, generator=gen) * 0.05).bfloat16().cuda()
    b = (torch.randn(g, n, k, generator=gen) * 0.05).bfloat16().cuda()
    d = (torch.randn(g, m, n, generator=gen) * 0.05).bfloat16().cuda()
    out = torch.empty(g, m, n, dtype=torch.bfloat16, device="cuda:0")
    out_t = torch.empty(g, n, m, dtype=torch.bfloat16, device="cuda:0")
    gram = torch.empty(g, m, m, dtype=torch.bfloat16, device="cuda:0")
    gemm_nt_batched(a, b, out, out_t=out_t, d_t=d.transpose(1, 2).contiguous(), alpha=0.7, beta=1.5)
    gram_batched(a.transpose(1, 2).contiguous(), gram)
    for i in range(g):
        one, two = torch.empty_like(out[i]), torch.empty_like(gram[i])
        gemm(a[i], b[i], True, one, d=d[i], alpha=0.7, beta=1.5)
        gemm(a[i], a[i], True, two)
        torch.cuda.synchronize()
        assert torch.equal(out[i].view(torch.int16), one.view(torch.int16))
        assert torch.equal(out_t[i].view(torch.int16), one.T.contiguous().view(torch.int16))
        assert torch.equal(gram[i].view(torch.int16), two.view(torch.int16))
