"""The attention kernels take the tiles of a large grid in an order of their own (whole layers of 256 workgroups, every second
one backwards).  A batch gives what its rows give in small grids, which are taken in plain order: the forward the same bits;
the backward too where both are two launches, else up to the order of the 64 additions in delta (a few 2^-24 of the
gradients, or now and then one rounding to bf16)."""
import pytest
import torch

from util import DTYPES, f64, gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("dtype", DTYPES)
# workgroups: 257 (no whole second layer), 512 (exactly two), 720, 540 with ragged last tiles, 1028 (four layers and a rest)
@pytest.mark.parametrize("B,H,T", [(257, 1, 64), (64, 4, 256), (30, 12, 256), (15, 12, 320), (257, 2, 192)])
@pytest.mark.parametrize("train", [False, True])
def test_attn_large_grid_against_rows(mt, dtype, B, H, T, train):
    g = gen(B + T)
    qkv = randn(g, B, H, 3, T, 64, dtype=dtype).to(DEV)
    dO = randn(g, B, H, T, 64, dtype=dtype).to(DEV)
    mask = torch.tril(torch.ones(T, T, dtype=torch.bool)).expand(B, T, T).contiguous().to(DEV)
    o, acts = mt.t_scaled_dot_prod_attn_fwd3_t(qkv, mask, train, 7)
    grads = mt.t_scaled_dot_prod_attn_bkwd3_t(dO, acts, qkv, mask, train, 7)
    n = max(1, 128 // (H * ((T + 127) // 128)))          # rows of at most half a layer
    tol = 2e-6 if dtype == torch.float32 else 2e-3
    for b in range(0, B, n):
        r = slice(b, b + n)
        part = mask[r].contiguous()
        o1, acts1 = mt.t_scaled_dot_prod_attn_fwd3_t(qkv[r].contiguous(), part, train, 7 + b * H)
        assert torch.equal(o1, o[r]) and torch.equal(acts1[0], acts[0][r]) and torch.equal(acts1[1], acts[1][r])
        small = mt.t_scaled_dot_prod_attn_bkwd3_t(dO[r].contiguous(), acts1, qkv[r].contiguous(), part, train, 7 + b * H)
        for got, want, what in zip(grads, small, ("dq", "dk", "dv")):
            x, y = f64(got[r]), f64(want)
            assert (x - y).norm() <= tol * y.norm(), (what, b)
