"""Q4_K with up to four lhs rows on many weight rows: five to eight tiles of 16 rows per workgroup, and more workgroups than compute units behind
that; one and two groups of K; against float64 products of the dequantised weights."""
import pytest
import torch

from mojo_amd import QuantizationEncoding as QE, dequantize, qmatmul, qmatmul_grouped, qmatmul_swiglu, quantize

pytestmark = pytest.mark.gpu


def packed(n, k):
    return quantize(QE.Q4_K, torch.empty((n, k), device="cuda").normal_(0.0, 0.02, generator=torch.Generator(device="cuda").manual_seed(n)))


def check(got, w, a):
    w, x = dequantize(QE.Q4_K, w).double(), a.double()
    # A lhs value is two fp16 terms cut toward zero (2^-21); K / 32 products enter a sum, then 8 wavefronts; a product is the difference of two
    # terms up to sixteen times as large (code and minimum).
    bound = (2.0**-21 + (a.shape[1] / 32 + 16) * 2.0**-24) * 16 * (x.abs() @ w.abs().T) + 1e-30
    worst = ((got.double() - x @ w.T).abs() / bound).max().item()
    assert worst <= 1.0, (got.shape, a.shape, worst)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(2, 16392, 4096), (3, 32768, 4096), (4, 32776, 4352), (4, 20488, 2304), (3, 24584, 4352)])
def test_many_tiles(m, n, k, lhs):
    w = packed(n, k)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
    a[m - 1] *= 1e-6
    check(qmatmul(QE.Q4_K, None, a, w), w, a)


def test_group_and_gated_pair():
    m, k, ns = 4, 4096, (14344, 14344, 40)
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(1))
    ws = [packed(n, k) for n in ns]
    outs = qmatmul_grouped(QE.Q4_K, a, ws)
    for got, w in zip(outs, ws):
        assert torch.equal(got, qmatmul(QE.Q4_K, None, a, w))
        check(got, w, a)
    gated = qmatmul_swiglu(QE.Q4_K, a, ws[0], ws[1]).double()
    want = torch.nn.functional.silu(outs[0].double()) * outs[1].double()
    assert torch.allclose(gated, want, rtol=1e-5, atol=1e-6)  # (exp and the quotient in fp32: some units of 2^-24 each)


@pytest.mark.parametrize("lhs", [torch.float32, torch.bfloat16])
@pytest.mark.parametrize("m,n,k", [(2, 4104, 4096), (3, 1032, 8448), (4, 14344, 256), (4, 32776, 2304), (5, 4104, 4352), (8, 20488, 512)])
def test_gated_pair_is_the_two_products_combined(m, n, k, lhs):
    gate, up = packed(n, k), packed(n + 8, k)[:n].contiguous()
    a = torch.randn((m, k), device="cuda", generator=torch.Generator(device="cuda").manual_seed(m)).to(lhs)
    products = qmatmul_grouped(QE.Q4_K, a, [gate, up])
    check(products[0], gate, a)
    check(products[1], up, a)
    g, u = (p.double() for p in products)
    # the same sums in the same order; exp, the quotient and two products in fp32 (8 units of 2^-24)
    assert torch.allclose(qmatmul_swiglu(QE.Q4_K, a, gate, up).double(), g / (1 + torch.exp(-g)) * u, rtol=2.0**-21, atol=1e-30)
