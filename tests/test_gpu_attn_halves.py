"""bf16 attention backward of small grids, where two wavefronts share a block of rows: against the grid that is large enough for every
wavefront to have a block of its own (the same rows many times), tile counts odd and even, masks that hide one half of a tile."""
import pytest
import torch

from util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("T", [128, 192, 256, 448, 1024])
@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("masked", [False, True])
def test_small_grid_against_large(mt, T, train, masked):
    g = gen(T)
    heads = 1024 // (2 * ((T + 127) // 128)) + 1     # more than four rounds of both backward passes: two launches
    q1, d1 = randn(g, 1, 1, 3, T, 64, dtype=torch.bfloat16).to(DEV), randn(g, 1, 1, T, 64, dtype=torch.bfloat16).to(DEV)
    doc = torch.bucketize(torch.arange(T), torch.tensor([24, 32, 70, T - 33]), right=True)
    seen = doc[:, None] == doc[None, :] if masked else torch.ones(T, T, dtype=torch.bool)
    if masked:
        seen &= (doc < 4)[:, None]                   # rows without a visible key
    mask = seen.tril()[None].contiguous().to(DEV) if masked else None
    # head 0 of the large grid has the small one's seed
    big, dbig = q1.expand(1, heads, 3, T, 64).contiguous(), d1.expand(1, heads, T, 64).contiguous()
    o1, a1 = mt.t_scaled_dot_prod_attn_fwd3_t(q1, mask, train, 3)
    o2, a2 = mt.t_scaled_dot_prod_attn_fwd3_t(big, mask, train, 3)
    pairs = [("o", o1[:, 0], o2[:, 0])] + [("ms", a1[0], a2[0][:, :1]), ("ls", a1[1], a2[1][:, :1])]
    g1 = mt.t_scaled_dot_prod_attn_bkwd3_t(d1, a1, q1, mask, train, 3)
    g2 = mt.t_scaled_dot_prod_attn_bkwd3_t(dbig, a2, big, mask, train, 3)
    pairs += [(n, x[:, 0], y[:, 0]) for n, x, y in zip(("dq", "dk", "dv"), g1, g2)]
    for what, x, y in pairs:
        x, y = x.double().flatten(), y.double().flatten()
        assert torch.isfinite(x).all(), what
        # both round P, dS and the result to bf16: 2^-9 each, in another order of sums
        assert (x - y).norm() <= 6e-3 * y.norm(), (what, ((x - y).norm() / y.norm()).item())
