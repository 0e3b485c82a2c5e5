"""fp32 products on the bf16 matrix pipe (three-way split operands): their error against fp64 stays below what
fp32 multiply-adds leave -- relative to sum_k |a b|, an rms of sqrt(K) roundings of 2^-24 for operands of one
sign, less for N(0,1) ones -- also where the operands' magnitudes differ by many orders."""
import pytest
import torch

from util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("n,m,k", [(1024, 3072, 768), (2048, 2304, 1000), (3000, 1032, 516), (768, 3072, 4100)])
@pytest.mark.parametrize("kind", ["normal", "positive", "wide"])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_error_is_below_fp32_accumulation(mt, n, m, k, kind, layout):
    g = gen(n + m + k)
    a, b = randn(g, n, k), randn(g, k, m)
    if kind == "positive":
        a, b = a.abs(), b.abs()
    if kind == "wide":      # magnitudes over some twelve orders
        a, b = a * torch.exp(3 * randn(g, n, k)), b * torch.exp(3 * randn(g, k, m))
    ad = a.to(DEV) if layout[0] == "n" else a.t().contiguous().to(DEV).t()
    bd = b.to(DEV) if layout[1] == "n" else b.t().contiguous().to(DEV).t()
    c = mt.matmul_t(ad, bd).double()
    a64, b64 = a.to(DEV).double(), b.to(DEV).double()
    err = (c - a64 @ b64) / (a64.abs() @ b64.abs())
    rms, worst = err.square().mean().sqrt().item(), err.abs().max().item()
    # what v_mfma_f32_32x32x2_f32 measures at K = 768: 1.4e-8 / 1.0e-7 / 1.3e-7 rms, growing with sqrt(K) where signs agree
    grow = max(1.0, (k / 768) ** 0.5)
    bar = {"normal": 1.45e-8 * max(1.0, (768 / k) ** 0.5), "positive": 1.05e-7 * grow, "wide": 1.35e-7 * grow}[kind]
    assert rms <= bar, (rms, bar)
    assert worst <= 12 * bar, (worst, bar)


def test_exact_where_fp32_is_exact(mt):
    """Small integers and powers of two: every product and partial sum is exact, so the result is too."""
    g = gen(3)
    a = torch.randint(-4095, 4096, (256, 512), generator=g).float()
    b = torch.ldexp(torch.ones(512, 256), torch.randint(0, 2, (512, 256), generator=g))
    c = mt.matmul_t(a.to(DEV), b.to(DEV))
    assert torch.equal(c.cpu().double(), a.double() @ b.double())


@pytest.mark.parametrize("n,m,k", [(512, 768, 768), (257, 131, 77), (96, 160, 2048)])
@pytest.mark.parametrize("b_t", [False, True])
def test_non_finite_operands(mt, n, m, k, b_t):
    """Infinities, NaN and values next to the largest float, which round to an infinite bf16 value, give what fp32
    multiply-adds give: the same classes as fp64, finite elements to fp32 accuracy."""
    g = torch.Generator().manual_seed(n)
    a, b = torch.randn(n, k, generator=g), torch.randn(m, k, generator=g) * 1e-3
    a[3, 5], a[7, 0], a[7, k - 1], a[n - 1, k // 2] = float("inf"), float("inf"), float("-inf"), float("nan")
    a[11, 2], a[12, k - 1] = 3.4e38, -3.4e38
    b[1, k - 2], b[m - 1, 9] = float("-inf"), 0.0
    want = a.double() @ b.double().t()
    bd = b.cuda().t() if b_t else b.t().contiguous().cuda()
    got = mt.t_matmul_t(a.cuda(), bd).double().cpu()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf = torch.isinf(want)
    assert torch.equal(got[inf], want[inf]) and torch.equal(torch.isinf(got), inf)
    fin = torch.isfinite(want)
    mag = torch.nan_to_num(a).double().abs() @ torch.nan_to_num(b).double().abs().t()
    # a chain of k multiply-adds: k 2^-24 of the summed magnitudes
    assert ((got - want).abs()[fin] <= (k * 2.0 ** -24 * mag)[fin]).all()
