"""The forward of few tokens with every norm inside the product that reads it against the forward that keeps its activations, whose
norms are launches of their own: tiles of 16 and of 32 rows, of 32 and of 64 columns (16x32, 16x64, 32x64 and, at 320 tokens, 32x32),
last tiles that are not whole in either direction, every width that is taken, one block and several, dense rows and partial sums, and
parameters off the 16-byte grid.  The same bits where the products alone take tiles with the same order of sums."""
import pytest
import torch

from oracle import gpt2 as ogpt2

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("D,F,L,B,T,shift", [(768, 3072, 2, 1, 64, 0), (768, 3072, 3, 1, 128, 0), (768, 2052, 2, 1, 64, 0), (768, 36, 2, 3, 64, 0),
                                             (256, 1024, 3, 1, 64, 0), (256, 1000, 2, 3, 64, 0), (512, 2048, 2, 1, 64, 0), (512, 2048, 2, 1, 192, 0),
                                             (1024, 1024, 2, 1, 64, 0), (1024, 4096, 2, 1, 64, 0), (768, 3072, 1, 1, 64, 0), (320, 1280, 2, 1, 64, 0),
                                             (768, 3072, 2, 1, 64, 1), (768, 800, 2, 5, 64, 0),
                                             (1024, 800, 2, 5, 64, 0), (768, 3072, 12, 1, 64, 0), (768, 3072, 12, 2, 64, 0)])
def test_norms_inside_products(mt, D, F, L, B, T, shift):
    V, H = 101, D // 64
    full = [[p.to(DEV) for p in grp] for grp in ogpt2.init_transformer_gpt2(V, D, L, H, F, T, seed=3)]
    gen = torch.Generator(device=DEV).manual_seed(5)
    for grp in full[2:]:
        for p in grp:
            if p.dim() == 1:
                p.add_(torch.randn(p.shape, generator=gen, device=DEV), alpha=0.1)
    params = [[p.to(torch.bfloat16) for p in grp] for grp in full]
    if shift:
        params[2][4] = torch.cat([params[2][4][:1], params[2][4]])[shift:]
        assert params[2][4].data_ptr() % 16 != 0
    y = torch.randint(0, V, (B, T), generator=torch.Generator().manual_seed(7)).to(DEV)
    exact = mt.t_gpt2_forward_t([[p.float() for p in grp] for grp in params], y, None, None, False).double()
    inside = mt.t_gpt2_forward_t(params, y, None, None, False)
    apart = mt.t_gpt2_forward_with_acts_t(params, y, None, None, False)[0]
    assert torch.isfinite(inside).all()
    if (D, F, B * T) not in ((512, 2048, 192), (1024, 800, 320)):         # (there the products alone take tiles of other K groups)
        assert torch.equal(inside.reshape(-1), apart.reshape(-1))
    # both round the same values to 2^-9, each tensor on the way of independent sign: errors of one size, which differ by how many
    # roundings fell otherwise
    err = [float((o.double().view(-1) - exact.view(-1)).norm() / exact.norm()) for o in (inside, apart)]
    assert err[0] <= 1.2 * err[1] and err[1] < 2e-2, err
