"""Products that share a launch (ptj_gemm_many) against fp64, under the bound of the single products: tiles that end inside in every
direction, contractions shorter than a step and not whole steps, outputs off the 16-byte grid, layouts and counts that go one by one."""
import ctypes
import importlib

import pytest
import torch

from util import DTYPES, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def operands(g, dtype, n, m, k, layout):
    a, b = randn(g, n, k).to(DEV).to(dtype), randn(g, k, m).to(DEV).to(dtype)
    return (a if layout[0] == "n" else a.t().contiguous().t(), b if layout[1] == "n" else b.t().contiguous().t())


def check(dtype, a, b, c):
    a64, b64 = a.double(), b.double()
    want, mag = a64 @ b64, a64.abs() @ b64.abs()
    # fp32: a rounding of 2^-24 per sixteen products and more; bf16: besides one rounding of the result, at most 2^-8 of it
    bound = 1e-5 * mag + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
    assert ((c.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("shapes", [
    [(768, 3072, 1000, "tn"), (3072, 768, 1000, "tn"), (1000, 768, 3072, "nn")],            # a feed-forward block's backward
    [(3072, 776, 777, "nn"), (768, 3072, 1501, "tn"), (1501, 1032, 3072, "nn"), (130, 136, 8, "nn")],
    [(1200, 1544, 40, "tn"), (1281, 1280, 72, "nn")],
    [(256, 512, 300, "nt"), (1536, 1536, 512, "tn")],                                       # a layout that goes one by one
    [(512, 512, 64, "nn")] * 5, [(512, 520, 64, "tn")], []])
def test_products_that_share_a_launch(mt, dtype, shapes):
    g = gen(len(shapes))
    pairs = [operands(g, dtype, *s) for s in shapes]
    if not pairs:
        lib = importlib.import_module("pre-tjax_amd")._lib
        assert lib.lib().ptj_gemm_many(None, 0, None, 0, 0, lib.stream()) == 0
        return
    for (a, b), c in zip(pairs, mt._matmul_many_t(*pairs)):
        check(dtype, a, b, c)


@pytest.mark.parametrize("dtype", DTYPES)
def test_outputs_off_the_grid(dtype):
    lib = importlib.import_module("pre-tjax_amd")._lib
    g = gen(5)
    pairs = [operands(g, dtype, 900, 1536, 768, "nn"), operands(g, dtype, 1536, 784, 904, "tn")]
    bufs = [torch.full((a.shape[0] * (b.shape[1] + 3) + 1,), 7.0, dtype=dtype, device=DEV) for a, b in pairs]
    outs = [x[1:].view(a.shape[0], -1)[:, :b.shape[1]] for x, (a, b) in zip(bufs, pairs)]
    f = []
    for (a, b), c in zip(pairs, outs):
        f += [a.data_ptr(), b.data_ptr(), c.data_ptr(), a.shape[0], b.shape[1], a.shape[1], a.stride(0), a.stride(1), b.stride(0),
              b.stride(1), c.stride(0)]
    p = (ctypes.c_int64 * len(f))(*f)
    lib.check(lib.lib().ptj_gemm_many(p, 2, None, 0, lib.dtype_code(bufs[0]), lib.stream()), "many")
    for (a, b), c, x in zip(pairs, outs, bufs):
        check(dtype, a, b, c)
        assert (x[1:].view(a.shape[0], -1)[:, b.shape[1]:] == 7.0).all() and x[0] == 7.0


@pytest.mark.parametrize("rows", [64, 500, 777, 1500, 3001, 6000])
@pytest.mark.parametrize("positive", [False, True])
def test_fp32_sums_are_no_less_exact_than_the_single_products(mt, rows, positive):
    """A feed-forward block's three products: a single one may be K-split, whose chains of additions are short."""
    g = gen(rows)
    shapes = [(768, 3072, rows, "tn"), (3072, 768, rows, "tn"), (rows, 768, 3072, "nn")]
    pairs = [operands(g, torch.float32, *s) for s in shapes]
    if positive:
        pairs = [(a.abs(), b.abs()) for a, b in pairs]
    for (a, b), c in zip(pairs, mt._matmul_many_t(*pairs)):
        want = a.double() @ b.double()
        error = [((x.double() - want).norm() / want.norm()).item() for x in (c, mt.matmul_t(a, b))]
        print("rows=%d %dx%d positive=%d: together %.3g, alone %.3g" % (rows, *c.shape, positive, *error))
        # two orders of the same roundings differ by chance, under 1 % over some 10^5 elements and more
        assert error[0] <= 1.01 * error[1]
