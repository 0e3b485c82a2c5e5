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


# Bars for N(0,1)-shaped operands from k = 8 on, relative to sum_k |a b|.  A model of the fp32 matrix instructions (two exact
# products and the accumulator per rounding) leaves 2.0e-8 rms and 2.2e-7 at worst over 4e5 elements at k = 8 .. 64 and less
# beyond; 2^-25 rms and 5 * 2^-24 at worst leave the hardware half a rounding more.  Results near the smallest fp32 number
# are rounded to multiples of 2^-149 besides, once per K split and once in their sum.
RMS, WORST, SMALLEST = 2.0 ** -25, 5 * 2.0 ** -24, 2.0 ** -149


@pytest.mark.parametrize("size_a,size_b", [(1e-35, 1e30), (1e-36, 1e29), (1e-37, 1e30), (1e-37, 1e35), (1e35, 1e-37), (1e-40, 1e31),
                                           (1e-42, 1e32), (1e-42, 1e36), (1e30, 1e-38), (1e-20, 1e-19), (1e12, 1e15), (1e17, 1e18)])
@pytest.mark.parametrize("n,m,k", [(1024, 3072, 768), (257, 131, 77), (640, 1031, 8)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
def test_operands_at_the_ends_of_the_range(mt, size_a, size_b, n, m, k, layout):
    """Tiny operands, subnormal ones among them, times large ones: the parts that a value is split into reach 24 binary
    orders below it, and what the split does not take is left to the fp32 instructions."""
    g = gen(k)
    a, b = (randn(g, n, k).double() * size_a).float().to(DEV), (randn(g, k, m).double() * size_b).float().to(DEV)
    ad = a if layout[0] == "n" else a.t().contiguous().t()
    bd = b if layout[1] == "n" else b.t().contiguous().t()
    c = mt.matmul_t(ad, bd).double()
    assert torch.isfinite(c).all()
    mag = a.double().abs() @ b.double().abs()
    err = ((c - a.double() @ b.double()).abs() - 2 * SMALLEST).clamp_min(0) / mag
    rms, worst = err.square().mean().sqrt().item(), err.max().item()
    assert rms <= RMS and worst <= WORST, (rms, worst)


@pytest.mark.parametrize("layout", ["nn", "tt"])
def test_magnitudes_mixed_inside_a_row(mt, layout):
    """Every row of A and column of B holds values over the whole range, and it is the tiny ones of one that meet the
    large ones of the other: a scale chosen by the largest value of a panel would lose them."""
    g = gen(12)
    n, m, k = 512, 1024, 96
    power = torch.randint(-140, 64, (k,), generator=g)
    a = (randn(g, n, k).double() * 2.0 ** power.double()).float().to(DEV)
    b = (randn(g, k, m).double() * 2.0 ** (-30 - power).clamp(max=90).double()[:, None]).float().to(DEV)
    ad = a if layout[0] == "n" else a.t().contiguous().t()
    bd = b if layout[1] == "n" else b.t().contiguous().t()
    c = mt.matmul_t(ad, bd).double()
    mag = a.double().abs() @ b.double().abs()
    err = (c - a.double() @ b.double()) / mag
    assert err.square().mean().sqrt().item() <= RMS and err.abs().max().item() <= WORST


@pytest.mark.parametrize("k", [8, 40])
def test_products_next_to_the_largest_float(mt, k):
    """A product below the largest float stays finite although the leading parts of its operands round up beyond it."""
    a, b = torch.zeros(136, k), torch.zeros(k, 265)
    a[:, k // 2] = 2.0 ** 64 * (1 - 2.0 ** -15)
    b[k // 2, :] = 2.0 ** 64 * (1 - 2.0 ** -15)
    c = mt.matmul_t(a.to(DEV), b.to(DEV)).cpu().double()
    want = a.double() @ b.double()
    assert torch.isfinite(c).all() and ((c - want).abs() <= 2.0 ** -24 * want).all()


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5])
def test_short_contractions(mt, k):
    """One product is rounded once, correctly; a few products leave at most one rounding each."""
    g = gen(k)
    a, b = randn(g, 301, 11).to(DEV)[:, :k], randn(g, k, 517).to(DEV)     # rows of 11: the split kernels take them
    c = mt.matmul_t(a, b).double()
    want = a.double() @ b.double()
    if k == 1:
        assert torch.equal(c, want.float().double())
    assert ((c - want).abs() <= k * 2.0 ** -24 * (a.double().abs() @ b.double().abs())).all()


def test_multiplying_epilogue_on_tiny_operands(mt):
    g = gen(21)
    a, b, mul = (randn(g, 1024, 96) * 1e-37).to(DEV), (randn(g, 96, 3072) * 1e30).to(DEV), randn(g, 1024, 3072).to(DEV)
    c, sums = mt.matmul_mul_colsum_t(a, b, mul)
    want, mag = (a.double() @ b.double()) * mul.double(), (a.double().abs() @ b.double().abs()) * mul.double().abs()
    assert ((c.double() - want).abs() <= WORST * mag + 2.0 ** -23 * want.abs()).all()
    # 1024 additions in fp32
    assert ((sums.double() - c.double().sum(0)).abs() <= 1024 * 2.0 ** -24 * c.double().abs().sum(0)).all()
