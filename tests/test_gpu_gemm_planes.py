"""fp32 products whose operands are split into three bf16 parts ahead of the product: sizes at which the size rule picks them, with
borders in every direction, an odd and an even number of steps, K splits, operands at any element alignment, values that the
split does not take, and the multiplying epilogue inside the native backward."""
import pytest
import torch

from oracle import gpt2 as ogpt2
from test_gpu_gemm_split import RMS, SMALLEST, WORST
from util import gen, randn, rel_l2

pytestmark = pytest.mark.gpu
DEV = "cuda"


def laid_out(x, transposed, shift):
    """x as a view of a buffer that starts `shift` elements behind a 16-byte boundary, rows three elements apart."""
    t = x.t() if transposed else x
    buf = torch.full((t.shape[0] * (t.shape[1] + 3) + shift,), float("nan"), device=DEV)
    v = buf[shift:].view(t.shape[0], t.shape[1] + 3)[:, :t.shape[1]]
    v.copy_(t)
    return v.t() if transposed else v


# N(0,1): the bars of the split products (what the fp32 instructions leave); the third: a K split
@pytest.mark.parametrize("n,m,k", [(4096, 3072, 768), (4001, 3079, 777), (3071, 3080, 4100)])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("shift", [0, 1])
def test_error_of_products_split_ahead(mt, n, m, k, layout, shift):
    g = gen(n + m + k)
    a, b, bias = randn(g, n, k).to(DEV), randn(g, k, m).to(DEV), randn(g, m).to(DEV)
    ad, bd = (laid_out(a, layout[0] == "t", shift), laid_out(b, layout[1] == "t", shift)) if shift else \
        (a if layout[0] == "n" else a.t().contiguous().t(), b if layout[1] == "n" else b.t().contiguous().t())
    c = mt.matmul_t(ad, bd, bias).double()
    mag = a.double().abs() @ b.double().abs() + bias.double().abs()
    err = (c - a.double() @ b.double() - bias.double()) / mag
    rms, worst = err.square().mean().sqrt().item(), err.abs().max().item()
    assert rms <= 1.45e-8 * max(1.0, (768 / k) ** 0.5) and worst <= 12 * 1.45e-8, (rms, worst)
    assert torch.equal(c, mt.matmul_t(ad, bd, bias).double())


@pytest.mark.parametrize("size_a,size_b", [(1e-37, 1e30), (1e-42, 1e36), (1e35, 1e-37), (1e17, 1e18)])
def test_range_of_products_split_ahead(mt, size_a, size_b):
    g = gen(7)
    n, m, k = 4096, 3072, 96
    a, b = (randn(g, n, k).double() * size_a).float().to(DEV), (randn(g, k, m).double() * size_b).float().to(DEV)
    c = mt.matmul_t(a, b).double()
    assert torch.isfinite(c).all()
    mag = a.double().abs() @ b.double().abs()
    err = ((c - a.double() @ b.double()).abs() - 2 * SMALLEST).clamp_min(0) / mag
    assert err.square().mean().sqrt().item() <= RMS and err.max().item() <= WORST


def test_non_finite_operands_split_ahead(mt):
    g = gen(8)
    n, m, k = 4001, 3079, 777
    a, b = randn(g, n, k).to(DEV), (randn(g, m, k) * 1e-3).to(DEV)
    a[3, 5], a[7, 0], a[7, k - 1], a[n - 1, k // 2] = float("inf"), float("inf"), float("-inf"), float("nan")
    a[1111, 2], b[1, k - 2], b[m - 1, 9] = 3.4e38, float("-inf"), 0.0
    got, want = mt.matmul_t(a, b.t()).double(), a.double() @ b.double().t()
    assert torch.equal(torch.isnan(got), torch.isnan(want))
    inf, fin = torch.isinf(want), torch.isfinite(want)
    assert torch.equal(got[inf], want[inf]) and torch.equal(torch.isinf(got), inf)
    mag = torch.nan_to_num(a).double().abs() @ torch.nan_to_num(b).double().abs().t()
    assert ((got - want).abs()[fin] <= (k * 2.0 ** -24 * mag)[fin]).all()


def test_native_backward_splits_ahead(mt, lo, monkeypatch):
    """2100 tokens (no whole tile): the native backward, whose scratch holds split operands also for the multiplying product,
    against the single calls, which form that one otherwise; both leave some 1e-7."""
    V, D, F, L, H, B, T = 101, 768, 3072, 1, 12, 7, 320
    params = [[p.to(DEV) for p in grp] for grp in ogpt2.init_transformer_gpt2(V, D, L, H, F, T, seed=3)]
    g = gen(9)
    y = torch.randint(1, V, (B, T + 1), generator=g).to(DEV)
    runs = []
    for native in (True, False):
        monkeypatch.setattr(mt, "NATIVE_STACK", native)
        runs.append(lo.t_loss_bkwd3_t(params, y, None, None, False, None)[0])
    for a, b in zip(sum((list(x) for x in runs[0]), []), sum((list(x) for x in runs[1]), [])):
        assert rel_l2(a, b.double().cpu()) <= 2e-6
