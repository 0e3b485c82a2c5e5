"""Products of operands whose rows start at any element (odd pitches, bases between vectors): sizes around the
tiles' edges, one-element remainders of every axis, and a K split; what lies around an operand is NaN and must not
reach the result."""
import pytest
import torch

from util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def _loose(x, transposed, pad, shift):
    """x as a view with a pitch of its width + pad, `shift` elements into a buffer of NaN."""
    t = x.t() if transposed else x
    rows, cols = t.shape
    buf = torch.full((shift + rows * (cols + pad) - pad,), float("nan"), dtype=x.dtype, device=DEV)
    v = buf.as_strided((rows, cols), (cols + pad, 1), shift)
    v.copy_(t)
    return v.t() if transposed else v


@pytest.mark.parametrize("dtype", [torch.bfloat16, torch.float32])
@pytest.mark.parametrize("layout", ["nn", "nt", "tn", "tt"])
@pytest.mark.parametrize("n,m,k", [(9, 11, 13), (1, 17, 9), (63, 65, 64), (64, 64, 65), (129, 127, 193), (127, 257, 321),
                                   (130, 70, 4099), (257, 1031, 515), (1025, 897, 1025)])
def test_any_pitch_and_base(mt, n, m, k, layout, dtype):
    g = gen(n * 7 + m * 5 + k)
    a, b, bias = randn(g, n, k).to(DEV, dtype), randn(g, k, m).to(DEV, dtype), randn(g, m + 1).to(DEV, dtype)[1:]
    pad = (0, 1) if (n * 1 + k) % 2 else (3, 5)
    av, bv = _loose(a, layout[0] == "t", pad[0], 1), _loose(b, layout[1] == "t", pad[1], 3)
    out = torch.full((n * (m + 3) + 1,), 7.0, dtype=dtype, device=DEV)
    c = mt.matmul_t(av, bv, bias, out=out[1:].as_strided((n, m), (m + 3, 1), 1))
    want = a.double() @ b.double() + bias.double()
    bound = 2e-7 * (a.double().abs() @ b.double().abs()) * max(1.0, (k / 64) ** 0.5) + (2.0 ** -8 if dtype == torch.bfloat16 else 1e-6) * want.abs() + 1e-6
    assert ((c.double() - want).abs() <= bound).all()
    rest = torch.ones_like(out, dtype=torch.bool)
    rest.as_strided((n, m), (m + 3, 1), 1).fill_(False)
    assert (out[rest] == 7.0).all()          # nothing is written outside C
