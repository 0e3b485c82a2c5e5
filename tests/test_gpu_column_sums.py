"""Second stages of column sums: the list kernel (a LayerNorm backward's dgamma, dbeta and the sums of its dropped output)
against fp64, at row counts around the 128 partial rows that a pass of it takes and on columns that fill no workgroup."""
import pytest
import torch

from util import DTYPES, f64, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 8, 257, 760, 8 * 127, 8 * 128 + 1, 8 * 225, 4095, 5000])
@pytest.mark.parametrize("cols", [72, 768])
def test_layernorm_column_sums(mt, dtype, rows, cols):
    g = gen(rows + cols)
    x, dy = randn(g, rows, cols, dtype=dtype), randn(g, rows, cols, dtype=dtype)
    ln = (randn(g, cols, dtype=dtype), randn(g, cols, dtype=dtype))
    dg, db = mt.t_layernorm_bkwd2_p_t(dy.to(DEV), tuple(p.to(DEV) for p in ln), x.to(DEV))
    xd, yd = f64(x), f64(dy)
    mu, sd = xd.mean(1, keepdim=True), xd.std(1, keepdim=True)
    xh = (xd - mu) / sd
    # fp32 sums of `rows` terms in chains of at most 40: 64 roundings of 2^-24 relative to the summed magnitudes, where a
    # term of dgamma counts with |x| + |mu| instead of their difference (mu and x - mu are rounded before the division);
    # bf16 results are rounded once (2^-8)
    for got, terms, mag in ((dg, yd * xh, (yd * (xd.abs() + mu.abs()) / sd).abs().sum(0)), (db, yd, yd.abs().sum(0))):
        want = terms.sum(0)
        bound = 64 * 2.0 ** -24 * mag + (2.0 ** -8 * want.abs() if dtype == torch.bfloat16 else 0)
        assert ((f64(got).reshape(-1) - want).abs() <= bound + 1e-30).all()
