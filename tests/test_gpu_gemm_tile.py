"""The one-tile-per-workgroup GEMM kernels: sizes at which the size rule picks each tile shape, with
border tiles, contraction lengths that end inside a 16-byte vector, K splits, and NaN in the pitch
padding of the operands (padding may be read but must not reach the result)."""
import pytest
import torch

from util import DTYPES, f64, gen, gemm_bound, randn
from oracle import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"

# few rows, one round of small tiles, wide outputs, half-filled large tiles, long contractions (K split)
SHAPES = [(1, 40, 19), (33, 72, 200), (64, 768, 768), (65, 776, 3075), (200, 2304, 770), (513, 3072, 768), (1000, 768, 3072),
          (3001, 768, 768), (768, 3072, 1001), (2304, 776, 3001), (3136, 3080, 768), (768, 768, 8195)]


def padded(x, dtype):
    """The same values in a buffer whose rows are padded to whole 16-byte vectors with NaN."""
    t = x if x.stride(1) == 1 else x.t()
    v = 16 // t.element_size()
    buf = torch.full((t.shape[0], (t.shape[1] + v - 1) // v * v), float("nan"), dtype=dtype, device=DEV)
    buf[:, :t.shape[1]] = t.to(DEV)
    r = buf[:, :t.shape[1]]
    return r if x.stride(1) == 1 else r.t()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,m,k", SHAPES)
@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
def test_tile_shapes(mt, dtype, n, m, k, layout):
    g = gen(n + 5 * m + 11 * k)
    a = randn(g, n, k, dtype=dtype) if layout[0] == "n" else randn(g, k, n, dtype=dtype).t()
    b = randn(g, k, m, dtype=dtype) if layout[1] == "n" else randn(g, m, k, dtype=dtype).t()
    bias = randn(g, m, dtype=dtype)
    ad, bd = padded(a, dtype), padded(b, dtype)
    v = 16 // ad.element_size()
    out = torch.full((n, (m + v - 1) // v * v), 7.0, dtype=dtype, device=DEV)
    aux = torch.empty_like(out)
    mt.matmul_t(ad, bd, bias.to(DEV), gelu=True, out=out[:, :m], deriv_out=aux[:, :m])
    a64, b64 = f64(a), f64(b)
    pre = a64 @ b64 + f64(bias)
    scale = a64.abs() @ b64.abs() + f64(bias).abs()
    want = ops.gelu(pre)
    assert ((f64(out[:, :m]) - want).abs() / gemm_bound(want, scale, dtype, 1.2)).max().item() <= 1.0
    assert (out[:, m:] == 7.0).all()                        # nothing is written past the last column
    x = pre.requires_grad_(True)
    ops.gelu(x).sum().backward()
    assert ((f64(aux[:, :m]) - x.grad).abs() / gemm_bound(x.grad, scale, dtype, 1.5)).max().item() <= 1.0
    c = mt.matmul_t(ad, bd)
    assert torch.equal(c, mt.matmul_t(ad, bd))              # K splits are reduced in fixed order


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("n,m,k", [(1, 40, 19), (65, 776, 768), (513, 3072, 768), (3001, 3080, 770)])
def test_tile_multiply_epilogue(mt, dtype, n, m, k):
    g = gen(n + m + k)
    a, b, mul = randn(g, n, k, dtype=dtype), randn(g, k, m, dtype=dtype), randn(g, n, m, dtype=dtype)
    ad, bd = padded(a, dtype), padded(b, dtype)
    c, sums = mt.matmul_mul_colsum_t(ad, bd, mul.to(DEV))
    want = (f64(a) @ f64(b)) * f64(mul)
    scale = (f64(a).abs() @ f64(b).abs()) * f64(mul).abs()
    assert ((f64(c) - want).abs() / (2 * gemm_bound(want, scale, dtype, 1.0))).max().item() <= 1.0
    cs = f64(c).sum(0)
    assert ((f64(sums) - cs).abs() / (1e-5 * f64(c).abs().sum(0) + 2.0 ** -8 * cs.abs() + 1e-6)).max().item() <= 1.0
