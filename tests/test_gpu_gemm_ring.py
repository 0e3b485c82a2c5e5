"""The persistent bf16 GEMM kernels: sizes at which the size rule picks them, so that workgroups walk one, two or three tiles of
either width, with borders in both directions, contraction lengths that end inside a step and inside a 16-byte vector, K splits,
a last round that is split, accumulation onto C from one step per tile up, and operands whose rows overlap."""
import importlib

import pytest
import torch

from test_gpu_gemm_tile import padded
from util import f64, gen, gemm_bound, randn
from oracle import ops

pytestmark = pytest.mark.gpu
DEV = "cuda"
BF16 = torch.bfloat16


def operands(n, m, k, layout, std=1.0):
    g = gen(n + 5 * m + 11 * k)
    a = randn(g, n, k, dtype=BF16, std=std) if layout[0] == "n" else randn(g, k, n, dtype=BF16, std=std).t()
    b = randn(g, k, m, dtype=BF16, std=std) if layout[1] == "n" else randn(g, m, k, dtype=BF16, std=std).t()
    return a, b, g


def product(a, b):
    """fp64 product and sum of magnitudes, on the GPU."""
    a64, b64 = a.to(DEV).double(), b.to(DEV).double()
    return (a64 @ b64).cpu(), (a64.abs() @ b64.abs()).cpu()


# 3001 x 3080: one partial round; 8200 x 3080: two; 16400 x 2305: three; the last two: K splits of few tiles
@pytest.mark.parametrize("n,m,k", [(3001, 3080, 770), (8200, 3080, 130), (16400, 2305, 200), (3079, 777, 8195), (2304, 768, 16384)])
@pytest.mark.parametrize("layout", ["nt", "nn", "tn", "tt"])
def test_ring_shapes(mt, n, m, k, layout):
    a, b, g = operands(n, m, k, layout)
    bias = randn(g, m, dtype=BF16)
    ad, bd = padded(a, BF16), padded(b, BF16)
    out = torch.full((n, (m + 15) // 8 * 8), 7.0, dtype=BF16, device=DEV)
    aux = torch.full_like(out, 7.0)
    mt.matmul_t(ad, bd, bias.to(DEV), gelu=True, out=out[:, :m], deriv_out=aux[:, :m])
    pre, scale = product(a, b)
    pre, scale = pre + f64(bias), scale + f64(bias).abs()
    want = ops.gelu(pre)
    assert ((f64(out[:, :m]) - want).abs() / gemm_bound(want, scale, BF16, 1.2)).max().item() <= 1.0
    x = pre.requires_grad_(True)
    ops.gelu(x).sum().backward()
    assert ((f64(aux[:, :m]) - x.grad).abs() / gemm_bound(x.grad, scale, BF16, 1.5)).max().item() <= 1.0
    assert (out[:, m:] == 7.0).all() and (aux[:, m:] == 7.0).all()
    c = mt.matmul_t(ad, bd)
    want, scale = product(a, b)
    assert ((f64(c) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0
    assert torch.equal(c, mt.matmul_t(ad, bd))
    odd = torch.full((n, m + 3), 7.0, dtype=BF16, device=DEV)      # rows of the output off the 16-byte grid
    mt.matmul_t(ad, bd, out=odd[:, 1:m + 1])
    assert ((f64(odd[:, 1:m + 1]) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0
    assert (odd[:, 0] == 7.0).all() and (odd[:, m + 1:] == 7.0).all()


# The walk over the tiles: every tile once where the tile rows are fewer than a group of four or leave a smaller last group, and the
# XCDs' ranges have different lengths (3 x 197, 9 x 49 and 5 x 33 tiles of 256 x 256, more columns at 192)
@pytest.mark.parametrize("n,m,k", [(700, 50257, 128), (2100, 12300, 128), (1100, 8200, 256)])
def test_ring_walk(mt, n, m, k):
    a, b, _ = operands(n, m, k, "nt")
    out = torch.full((n, (m + 15) // 8 * 8), 7.0, dtype=BF16, device=DEV)
    mt.matmul_t(padded(a, BF16), padded(b, BF16), out=out[:, :m])
    want, scale = product(a, b)
    assert ((f64(out[:, :m]) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0
    assert (out[:, m:] == 7.0).all()


# one shape for each kernel that forms the derivative: ring, tiles, K split, unaligned and strided operands, fp32 tiles, fp32 split
# per tile and ahead
@pytest.mark.parametrize("n,m,k,dtype,step", [(3001, 3080, 128, BF16, 1), (100, 776, 64, BF16, 1), (64, 768, 4096, BF16, 1),
                                              (100, 771, 65, BF16, 1), (100, 776, 64, BF16, 2), (70, 128, 64, torch.float32, 1),
                                              (512, 768, 256, torch.float32, 1), (4096, 3072, 128, torch.float32, 1)])
def test_gelu_derivative_of_large_preactivations(mt, n, m, k, dtype, step):
    """Pre-activations over the whole finite range: the GELU is x or 0 and its derivative exactly 1 or 0."""
    g = gen(n + m + k)
    a, b = randn(g, n, k * step, dtype=dtype, std=0.1).to(DEV)[:, ::step], randn(g, k, m, dtype=dtype, std=0.1).to(DEV)
    big = torch.tensor([64.0, 1e3, 1.1e13, 1.3e13, 1e15, 1.7e19, 2e19, 1e30, 3.3e38])
    bias = torch.cat([big, -big]).repeat(m // 18 + 1)[:m].to(dtype).to(DEV)
    out, deriv = (torch.empty(n, m, dtype=dtype, device=DEV) for _ in range(2))
    mt.matmul_t(a, b, bias, gelu=True, out=out, deriv_out=deriv)
    pos = (bias > 0).expand(n, m)
    assert torch.equal(deriv, pos.to(dtype))
    x = mt.matmul_t(a, b, bias)
    assert torch.equal(out, torch.where(pos, x, torch.zeros_like(x)))


@pytest.mark.parametrize("n,m,k", [(3001, 3080, 770), (16400, 3076, 128)])
@pytest.mark.parametrize("layout", ["nn", "tt"])
def test_ring_multiply_epilogue(mt, n, m, k, layout):
    a, b, g = operands(n, m, k, layout)
    mul = randn(g, n, m, dtype=BF16)
    c, sums = mt.matmul_mul_colsum_t(padded(a, BF16), padded(b, BF16), mul.to(DEV))
    want, scale = product(a, b)
    want, scale = want * f64(mul), scale * f64(mul).abs()
    assert ((f64(c) - want).abs() / (2 * gemm_bound(want, scale, BF16, 1.0))).max().item() <= 1.0
    cs = f64(c).sum(0)
    assert ((f64(sums) - cs).abs() / (1e-5 * f64(c).abs().sum(0) + 2.0 ** -8 * cs.abs() + 1e-6)).max().item() <= 1.0


@pytest.mark.parametrize("n,m,k", [(300, 520, 64), (8, 8, 128), (20001, 776, 192), (257, 193, 1024)])
@pytest.mark.parametrize("layout", ["nn", "tn", "tt"])
def test_ring_accumulates(mt, n, m, k, layout):
    a, b, g = operands(n, m, k, layout)
    out = torch.full((n, (m + 7) // 8 * 8), 7.0, dtype=BF16, device=DEV)
    c0 = randn(g, n, m, dtype=BF16)
    out[:, :m] = c0.to(DEV)
    mt.matmul_t(padded(a, BF16), padded(b, BF16), out=out[:, :m], accumulate=True)
    want, scale = product(a, b)
    want, scale = want + f64(c0), scale + f64(c0).abs()
    assert ((f64(out[:, :m]) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0
    assert (out[:, m:] == 7.0).all()


@pytest.mark.parametrize("k", [64, 192, 130])
def test_ring_rows_that_overlap(mt, k):
    """One row for all of A, windows of one buffer as B's rows."""
    n, m = 3000, 776
    g = gen(k)
    a = randn(g, 1, k, dtype=BF16).to(DEV).expand(n, k)
    b = randn(g, m * 8 + k, dtype=BF16).to(DEV).as_strided((m, k), (8, 1)).t()
    c = mt.matmul_t(a, b)
    want, scale = product(a, b)
    assert ((f64(c) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0


def test_ring_rows_far_apart(mt):
    """Outputs and multipliers in column slices of buffers so wide that a lane's row leaves 32-bit offsets (the first 64 x 96 are
    a wavefront's whole block)."""
    n, m, k, pitch, at = 72, 136, 64, 150_000_000, 1_000_000
    g = gen(n)
    wide = torch.zeros(n, pitch, dtype=BF16, device=DEV)
    part = wide[:, at:at + m]
    a, b = randn(g, k, n, dtype=BF16).to(DEV).t(), randn(g, k, m, dtype=BF16).to(DEV)
    c0 = randn(g, n, m, dtype=BF16).to(DEV)
    part.copy_(c0)
    mt.matmul_t(a, b, out=part, accumulate=True)
    want = c0.clone()
    mt.matmul_t(a, b, out=want, accumulate=True)
    assert torch.equal(part, want) and torch.count_nonzero(wide) == torch.count_nonzero(part)
    # one row for all of A: operands that only these kernels take
    row = randn(g, 1, k, dtype=BF16).to(DEV).expand(n, k)
    bias, deriv = randn(g, m, dtype=BF16).to(DEV), torch.zeros_like(wide)
    mt.matmul_t(row, b, bias, gelu=True, out=part, deriv_out=deriv[:, at:at + m])
    out, d = torch.empty_like(c0), torch.empty_like(c0)
    mt.matmul_t(row, b, bias, gelu=True, out=out, deriv_out=d)
    assert torch.equal(part, out) and torch.equal(deriv[:, at:at + m], d)
    assert torch.count_nonzero(wide) == torch.count_nonzero(part) and torch.count_nonzero(deriv) == torch.count_nonzero(d)
    part.copy_(c0)
    c, sums = mt.matmul_mul_colsum_t(row, b, c0)
    for x, y in zip(mt.matmul_mul_colsum_t(row, b, part), (c, sums)):
        assert torch.equal(x, y)
    _lib = importlib.import_module("pre-tjax_amd._lib")
    ws = torch.empty(_lib.lib().ptj_gemm_mul_colsum_workspace_bytes(n, m), dtype=torch.uint8, device=DEV)
    sums2 = torch.empty_like(sums)
    _lib.check(_lib.lib().ptj_gemm_mul_colsum(row.data_ptr(), b.data_ptr(), c0.data_ptr(), part.data_ptr(), sums2.data_ptr(), n, m, k,
                                              *row.stride(), *b.stride(), m, pitch, ws.data_ptr(), ws.numel(), _lib.PTJ_BF16,
                                              _lib.stream()), "ptj_gemm_mul_colsum")
    assert torch.equal(part, c) and torch.equal(sums2, sums) and torch.count_nonzero(wide) == torch.count_nonzero(c)


def test_ring_contraction_rows_far_apart(mt):
    """A contraction of fewer indices than a step, its rows so far apart that those past the end leave 32-bit offsets."""
    n, m, k, pitch = 40, 136, 16, 50_000_000
    g = gen(k)
    a = randn(g, n, k, dtype=BF16).to(DEV)
    b = torch.full((k, pitch), float("nan"), dtype=BF16, device=DEV)[:, :m]
    b.copy_(randn(g, k, m, dtype=BF16).to(DEV))
    want, scale = product(a, b)
    assert ((f64(mt.matmul_t(a, b)) - want).abs() / gemm_bound(want, scale, BF16)).max().item() <= 1.0
