"""LayerNorm, forward and backward, and the residual update in front of it, at widths that every thread holds whole vectors of and at
those next to them."""
import pytest
import torch

from util import DTYPES, f64, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("cols", [256, 264, 504, 512, 520, 760, 768, 776, 1024, 1032, 2040, 2048])
@pytest.mark.parametrize("rows", [1, 9, 515])
def test_norm_widths(mt, dtype, cols, rows):
    g = gen(rows + cols)
    x, dy = randn(g, rows, cols, dtype=dtype).to(DEV), randn(g, rows, cols, dtype=dtype).to(DEV)
    res = randn(g, rows, cols, dtype=dtype).to(DEV)
    gamma, beta = randn(g, cols, dtype=dtype).to(DEV), randn(g, cols, dtype=dtype).to(DEV)
    # sums of `cols` (or `rows`) terms in fp32, rounded once to the storage type
    tol = 1e-5 if dtype == torch.float32 else 2.0 ** -7

    def close(a, want):
        assert (f64(a) - want).abs().max() <= tol * (1.0 + want.abs().max())

    y, h, _ = mt.dropout_add_layernorm_t(x, res, (gamma, beta), False, 3)
    assert torch.equal(y, mt.dropout_add_t(x, res, False, 3))
    for out, src in ((h, y), (mt.t_layernorm_fwd_t((gamma, beta), x), x)):
        s = f64(src)
        xh = (s - s.mean(1, keepdim=True)) / s.std(1, keepdim=True)
        close(out, xh * f64(gamma) + f64(beta))
    s = f64(x).requires_grad_()
    w, b = f64(gamma).requires_grad_(), f64(beta).requires_grad_()
    ((s - s.mean(1, keepdim=True)) / s.std(1, keepdim=True) * w + b).backward(f64(dy))
    close(mt.t_layernorm_bkwd2_x_t(dy, (gamma, beta), x), s.grad)
    dg, db = mt.t_layernorm_bkwd2_p_t(dy, (gamma, beta), x)
    close(dg, w.grad)
    close(db, b.grad)
