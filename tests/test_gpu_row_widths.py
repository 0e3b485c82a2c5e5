"""LayerNorm, forward and backward, and the residual update in front of it, at widths that every thread holds whole vectors of and at
those next to them."""
import pytest
import torch

from oracle import gpt2 as ogpt2
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


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("rows", [1, 7, 8, 9, 515, 4097])
def test_pipelined_backward_gives_the_bits_of_the_general_one(mt, dtype, rows):
    """768 columns: where the dropout decisions are read, or none are wanted, the next row is requested ahead; where they are formed anew
    the general kernel runs.  Everything but the dropped copy is the same either way, and the decisions are."""
    cols, seed = 768, 77
    g = gen(rows)
    x, dy, res = (randn(g, rows, cols, dtype=dtype).to(DEV) for _ in range(3))
    ln = randn(g, cols, dtype=dtype).to(DEV), randn(g, cols, dtype=dtype).to(DEV)
    zero = torch.zeros(rows, cols, dtype=torch.bfloat16, device=DEV)
    keep = mt.dropout_add_t(zero, zero, True, seed, want_keep=True)[1]
    for residual in (None, res):
        dx, (dg, db), dropped, dsum = mt.layernorm_bkwd2_t(dy, ln, x, residual=residual, drop=(True, seed), drop_sum=True)
        runs = [mt.layernorm_bkwd2_t(dy, ln, x, residual=residual)]
        if dtype == torch.bfloat16:          # (fp32 reads decisions in the native stack alone)
            runs.append(mt.layernorm_bkwd2_t(dy, ln, x, residual=residual, drop=(True, seed, keep), drop_sum=True))
            assert torch.equal(runs[1][2], dropped) and torch.equal(runs[1][3], dsum)
        for got in runs:
            assert torch.equal(got[0], dx) and torch.equal(got[1][0], dg) and torch.equal(got[1][1], db)


@pytest.mark.parametrize("B,T", [(1, 64), (3, 128), (1, 576)])
def test_fp32_backward_with_recorded_decisions(mt, lo, monkeypatch, B, T):
    """One block 768 wide: the native stack records the decisions of its dropouts and reads them in the pipelined kernel, the single calls
    form them anew in the general one."""
    params = [[p.to(DEV) for p in grp] for grp in ogpt2.init_transformer_gpt2(101, 768, 1, 12, 3072, T, seed=3)]
    y = torch.randint(0, 101, (B, T + 1), generator=torch.Generator().manual_seed(7)).to(DEV)
    runs = []
    for native in (True, False):
        monkeypatch.setattr(mt, "NATIVE_STACK", native)
        grads, _ = lo.t_loss_bkwd3_t(params, y, None, None, True, [10, 11, 12, 13])
        runs.append([p for grp in grads for p in grp])
    for i, (a, b) in enumerate(zip(*runs)):
        assert torch.equal(a, b), i
