"""The launch that forms the weight gradients of several blocks, by itself: against fp64 and against the single products, with
contractions of one step, of many and of a last step that is not whole, and with null operands."""
import ctypes
import importlib

import pytest
import torch

from util import DTYPES, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"
KINDS, BLOCKS = 4, 16


class Group(ctypes.Structure):          # csrc/internal.h: PtjGradGroup
    _fields_ = [("k", ctypes.c_int), ("blocks", ctypes.c_int), ("n", ctypes.c_int * KINDS), ("m", ctypes.c_int * KINDS),
                ("d", ctypes.c_void_p * BLOCKS * KINDS), ("x", ctypes.c_void_p * BLOCKS * KINDS),
                ("dw", ctypes.c_void_p * BLOCKS * KINDS)]


def launch(group, dtype):
    lib = importlib.import_module("pre-tjax_amd")._lib
    fn = getattr(lib.lib(), "_Z16ptj_weight_gradsRK12PtjGradGroupiP12ihipStream_t")
    fn.argtypes, fn.restype = [ctypes.c_void_p, ctypes.c_int, ctypes.c_void_p], ctypes.c_int
    return fn(ctypes.addressof(group), lib.dtype_code(torch.empty(0, dtype=dtype)), lib.stream())


def weight_gradients(dtype, k, blocks, shapes, scale=1.0):
    """operands and results of one launch: [(d [k, n], x [k, m], dw [n, m])], kinds inside blocks"""
    g, group, tensors = gen(k + blocks), Group(), []
    group.k, group.blocks = k, blocks
    for block in range(blocks):
        for kind, (n, m) in enumerate(shapes):
            group.n[kind], group.m[kind] = n, m
            d, x = (randn(g, k, n) * scale).to(DEV).to(dtype), randn(g, k, m).to(DEV).to(dtype)
            dw = torch.full((n * m + 64,), 7.0, dtype=dtype, device=DEV)
            group.d[kind][block], group.x[kind][block], group.dw[kind][block] = d.data_ptr(), x.data_ptr(), dw.data_ptr()
            tensors.append((d, x, dw))
    assert launch(group, dtype) == 0
    out = []
    for i, (d, x, dw) in enumerate(tensors):
        n, m = shapes[i % KINDS]
        assert (dw[n * m:] == 7.0).all()
        out.append((d, x, dw[:n * m].view(n, m)))
    return out


SMALL = [(320, 1288), (1288, 320), (320, 320), (960, 320)]
GPT2 = [(768, 3072), (3072, 768), (768, 768), (2304, 768)]


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("k", [1, 3, 64, 100, 129, 1000, 1024, 1025, 1055, 2081])
def test_every_length_of_the_contraction(dtype, k):
    for d, x, dw in weight_gradients(dtype, k, 8, SMALL):
        d, x = d.double(), x.double()
        want, mag = d.t() @ x, d.t().abs() @ x.abs()
        # as for the single products: a rounding of 2^-24 per sixteen products and more; bf16: besides, one of the result
        bound = 1e-5 * mag + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
        assert ((dw.double() - want).abs() <= bound).all()


@pytest.mark.parametrize("k", [64, 448, 1024, 1088, 1536, 2048, 4096])
@pytest.mark.parametrize("positive", [False, True])
def test_fp32_sums_are_no_less_exact_than_the_single_products(mt, k, positive):
    """A product on its own takes a K split from 1024 elements on, whose chains of additions are short; a tile of the group goes along the
    whole contraction."""
    for d, x, dw in weight_gradients(torch.float32, k, 2, GPT2)[:KINDS]:
        if positive:                   # sums as large as their terms allow
            group = Group()
            d, x = d.abs_(), x.abs_()
            group.k, group.blocks = k, 1
            for kind in range(KINDS):
                group.n[kind], group.m[kind] = d.shape[1], x.shape[1]
                out = dw if kind == 0 else torch.empty_like(dw)
                group.d[kind][0], group.x[kind][0], group.dw[kind][0] = d.data_ptr(), x.data_ptr(), out.data_ptr()
            assert launch(group, torch.float32) == 0
        want = d.double().t() @ x.double()
        error = [((c.double() - want).norm() / want.norm()).item() for c in (dw, mt.matmul_t(d.t(), x))]
        print("k=%d %dx%d positive=%d: together %.3g, alone %.3g" % (k, dw.shape[0], dw.shape[1], positive, *error))
        # two orders of the same roundings differ by chance, under 1 % over some 10^6 elements
        assert error[0] <= 1.01 * error[1]


def test_values_that_leave_the_split():
    """Sums from 2^96 on are formed again by the fp32 instructions."""
    for d, x, dw in weight_gradients(torch.float32, 1100, 2, SMALL, scale=2.0 ** 100):
        d, x = d.double(), x.double()
        assert ((dw.double() - d.t() @ x).abs() <= 1e-5 * (d.t().abs() @ x.abs())).all()


@pytest.mark.parametrize("field", ["d", "x", "dw"])
def test_null_operands_are_refused(field):
    group = Group()
    group.k, group.blocks = 64, 2
    for kind, (n, m) in enumerate(GPT2):
        group.n[kind], group.m[kind] = n, m
        for block in range(2):
            for f in ("d", "x", "dw"):
                getattr(group, f)[kind][block] = 0x1000
    getattr(group, field)[3][1] = None
    assert launch(group, torch.float32) == -1
