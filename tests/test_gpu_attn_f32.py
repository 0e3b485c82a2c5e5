"""fp32 attention on the bf16 matrix pipe: every factor is split into three bf16 values.  Against fp64, at the edges of the
tiles and of what the split covers."""
import pytest
import torch

from util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


def case(B, H, T, seed):
    g = gen(seed)
    qkv, do = randn(g, B, H, 3, T, 64).to(DEV), randn(g, B, H, T, 64).to(DEV)
    # documents that end inside a 32-row block, at its end and inside the next one, and a padded tail
    doc = torch.bucketize(torch.arange(T), torch.tensor([24, 32, 70, T - 9]), right=True)
    mask = torch.tril(doc[:, None] == doc[None, :]) & (doc < 4)[:, None] & (doc < 4)[None, :]
    return qkv, do, mask.expand(B, T, T).contiguous().to(DEV)


def both(mt, qkv, do, mask, train=False):
    o, acts = mt.t_scaled_dot_prod_attn_fwd3_t(qkv, mask, train, 3)
    return (o,) + tuple(mt.t_scaled_dot_prod_attn_bkwd3_t(do, acts, qkv, mask, train, 3))


def exact(qkv, do, mask):
    q, k, v = (qkv[:, :, i].double().cpu().requires_grad_() for i in range(3))
    s = (q @ k.transpose(-1, -2) / 8).masked_fill(~mask.cpu()[:, None], -1e9)
    o = 0.9 * torch.softmax(s, -1) * mask.cpu().any(-1)[:, None, :, None] @ v
    return [x.detach() for x in (o,) + torch.autograd.grad(o, (q, k, v), do.double().cpu())]


@pytest.mark.parametrize("B,H,T", [(1, 1, 64), (2, 1, 128), (1, 3, 192), (1, 2, 448)])
@pytest.mark.parametrize("masked", [False, True])
def test_error_against_fp64(mt, B, H, T, masked):
    """A score of 64 products is rounded 24 times, a sum over T keys 6 T / 16 times, by 2^-24 / sqrt(3) of its largest partial
    sum each; up to T = 448 these walks stay below 2^-24 sqrt(24 + 168) / sqrt(3) = 4.8e-7, and a factor of 2 covers P and dS,
    which carry the errors of the scores.  Two parts of a factor in place of three leave 2^-17."""
    qkv, do, mask = case(B, H, T, T)
    if not masked:
        mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril().expand(B, T, T).contiguous()
    for got, want, what in zip(both(mt, qkv, do, mask), exact(qkv, do, mask), ("o", "dq", "dk", "dv")):
        assert (got.double().cpu() - want).norm() <= 1e-6 * want.norm(), what


@pytest.mark.parametrize("T", [64, 192])
def test_both_directions_form_the_same_scores(mt, T):
    """Every query sees its own key alone, so P is 1 and dV = 0.9 dO, whatever the score.  The scores are sums of terms of a thousand that
    nearly cancel: formed in another order in the backward than in the forward they would differ by 1e-4 and more, and P with them.
    As the same bits they leave the rounding of the saved maximum (0.1), 1 / l, 0.9 P and the product: under 8 of 2^-24."""
    g = gen(T)
    q, v, do = (randn(g, 1, 2, T, 64) for _ in range(3))
    k = randn(g, 1, 2, T, 64)
    q, k = q * 30, k * 30
    # the last column takes what is left of the score but for about 0.3
    k[..., 63] = (0.3 - (q[..., :63].double() * k[..., :63].double()).sum(-1)).div(q[..., 63].double()).float()
    qkv = torch.stack([q, k, v], 2).to(DEV)
    mask = torch.eye(T, dtype=torch.bool, device=DEV)[None]
    _, dq, dk, dv = both(mt, qkv, do.to(DEV), mask)
    want = 0.9 * do.double()
    assert ((dv.double().cpu() - want).abs() <= 8 * 2.0 ** -24 * want.abs()).all()


@pytest.mark.parametrize("train", [False, True])
def test_gradients_scale_exactly(mt, train):
    """Every gradient is linear in dO: with dO a power of two smaller all parts, products and sums are, too."""
    qkv, do, mask = case(1, 2, 192, 5)
    a, b = both(mt, qkv, do, mask, train), both(mt, qkv, do * 2.0 ** -60, mask, train)
    assert all(torch.equal(x * 2.0 ** -60, y) for x, y in zip(a[1:], b[1:]))


@pytest.mark.parametrize("T", [64, 192])
@pytest.mark.parametrize("train", [False, True])
@pytest.mark.parametrize("masked", [False, True])
def test_values_that_are_not_split(mt, T, train, masked):
    """V from 2^32 on is multiplied by the fp32 instructions: O and the gradients of Q and K are as many times larger, that of V the
    same, but for what either way rounds (1e-6 each as in test_error_against_fp64)."""
    qkv, do, mask = case(2, 2, T, 7)
    if not masked:
        mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril().expand(2, T, T).contiguous()
    big = qkv.clone()
    big[:, :, 2] *= 2.0 ** 40
    for what, x, y, e in zip(("o", "dq", "dk", "dv"), both(mt, big, do, mask, train), both(mt, qkv, do, mask, train), (40, 40, 40, 0)):
        x, y = x.double() * 2.0 ** -e, y.double()
        assert torch.isfinite(x).all() and (x - y).norm() <= 2e-6 * y.norm(), what


def test_sharp_scores_against_the_fp32_instructions(mt):
    """Scores of nine times the size, whose rounding is what the results' error comes from: 32 roundings of a sum of 64 by the fp32
    instructions (which take V from 2^32 on), four at full size here.  0.35 of the error as a random walk; 0.6 leaves room for
    the roundings that both share, and not for six a chunk (24: 0.87)."""
    T = 192
    qkv, do, _ = case(4, 12, T, 12)
    qkv[:, :, :2] *= 3
    mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril().expand(4, T, T).contiguous()
    want = exact(qkv, do, mask)
    big = qkv.clone()
    big[:, :, 2] *= 2.0 ** 40
    for what, x, y, z, e in zip(("o", "dq", "dk", "dv"), both(mt, qkv, do, mask), both(mt, big, do, mask), want, (40, 40, 40, 0)):
        error = [(v.double().cpu() - z).norm().item() for v in (x, y.double() * 2.0 ** -e)]
        assert error[0] <= 0.6 * error[1], (what, error)


@pytest.mark.parametrize("train", [False, True])
def test_tiny_factors(mt, train):
    """Values of 2^-112, whose lowest parts are below bf16's range unless they are scaled.  Results are linear in V and dO, and with both a
    power of two smaller they are the same but for roundings below 2^-149 (subnormal ones, of products and of results): 2^-37 of
    the results each, a few of them a result."""
    qkv, do, mask = case(1, 2, 192, 9)
    small = qkv.clone()
    small[:, :, 2] *= 2.0 ** -112
    a, b = both(mt, qkv, do, mask, train), both(mt, small, do, mask, train)
    c = both(mt, qkv, do * 2.0 ** -112, mask, train)
    for what, x, y in [("o", b[0], a[0]), ("dq", b[1], a[1]), ("dk", b[2], a[2])] + [("do: " + n, x, y) for n, x, y in zip(("dq", "dk", "dv"), c[1:], a[1:])]:
        assert (x.double() * 2.0 ** 112 - y.double()).norm() <= 2.0 ** -30 * y.double().norm(), what


def test_tiny_probabilities(mt):
    """Every query sees key 0, whose V is 0, and itself with a score 80 lower: O is one product of P = 2^-115, dV of the key one as well.
    The scores have few bits, so the fp32 instructions (which take V from 2^32 on) multiply the same P where key 0 is in the same 32
    keys (elsewhere two partial results are put together, whose reference points are rounded)."""
    T = 128
    g = gen(10)
    qkv, do = torch.zeros(1, 1, 3, T, 64), randn(g, 1, 1, T, 64)
    qkv[:, :, 2, 1:] = randn(g, T - 1, 64)
    qkv[:, :, 0, :, 0], qkv[:, :, 1, 1:, 0] = 32.0, -20.0
    mask = torch.eye(T, dtype=torch.bool)
    mask[:, 0] = True
    mask, big = mask[None].to(DEV), qkv.clone()
    big[:, :, 2] *= 2.0 ** 40
    x, y = both(mt, qkv.to(DEV), do.to(DEV), mask), both(mt, big.to(DEV), do.to(DEV), mask)
    for what, got, want, n in (("o", x[0].double() * 2.0 ** 40, y[0].double(), 32), ("dv", x[3].double(), y[3].double(), T)):
        got, want = got[:, :, 1:n], want[:, :, 1:n]
        assert (want != 0).all() and ((got - want).abs() <= 3 * 2.0 ** -24 * want.abs() + 2.0 ** -148).all(), what


def test_infinite_factors(mt):
    """inf * -inf is -inf: key 10 is as good as hidden from every query, and so is every key from query 70."""
    T = 192
    qkv, do, _ = case(1, 1, T, 6)
    qkv[0, 0, 0, :, 3] = qkv[0, 0, 0, :, 3].abs()
    qkv[0, 0, 1, :, 3] = -qkv[0, 0, 1, :, 3].abs()
    mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()[None].contiguous()
    mask[:, :, 10] = False
    mask[:, 70] = False
    want = both(mt, qkv, do, mask)[0]
    qkv[0, 0, 0, 70, 3], qkv[0, 0, 1, 10, 3] = float("inf"), float("-inf")
    got = both(mt, qkv, do, torch.ones_like(mask).tril())[0]
    assert torch.equal(got[0, 0, 70], torch.zeros(64, device=DEV)) and (got - want).norm() <= 2e-6 * want.norm()


def test_overflowing_products_of_the_backward(mt):
    """dP of the last query and key 5 overflows, all else is finite: dQ of that query and dK of that key are infinite, with the signs
    of K and Q."""
    T = 64
    qkv, do, _ = case(1, 1, T, 8)
    qkv[0, 0, 2, :, 0], qkv[0, 0, 2, 5, 0] = 0.1, 2.0
    do[0, 0, T - 1], do[0, 0, T - 1, 0] = 0.0, 3e38
    _, dq, dk, dv = (x[0, 0] for x in both(mt, qkv, do, torch.ones(T, T, dtype=torch.bool, device=DEV).tril()[None]))
    q, k = qkv[0, 0, 0], qkv[0, 0, 1]
    assert torch.equal(dq[T - 1], float("inf") * k[5].sign()) and torch.equal(dk[5], float("inf") * q[T - 1].sign())
    rest = torch.ones(T, dtype=torch.bool, device=DEV)
    rest[5] = False
    assert torch.isfinite(dv).all() and torch.isfinite(dq[:T - 1]).all() and torch.isfinite(dk[rest]).all()


def test_large_and_infinite_values(mt):
    T = 192
    qkv, do, mask = case(1, 1, T, 6)
    mask = torch.ones(T, T, dtype=torch.bool, device=DEV).tril()[None]
    plain = both(mt, qkv, do, mask)[0]
    big = qkv.clone()
    big[:, :, 2] *= 2.0 ** 121
    got = both(mt, big, do, mask)[0]
    assert (got.double() * 2.0 ** -121 - plain.double()).norm() <= 1e-6 * plain.double().norm()
    inf = qkv.clone()
    inf[0, 0, 2, 70, 5], inf[0, 0, 2, 130, 9] = float("inf"), float("-inf")
    got = both(mt, inf, do, mask)[0][0, 0]
    assert torch.isposinf(got[70:, 5]).all() and torch.isneginf(got[130:, 9]).all()
    # (a hidden key's probability is 0 and 0 * inf is NaN where its tile is visited, as it was with fp32 products)
    clean = torch.ones_like(got, dtype=torch.bool)
    clean[:, 5] = clean[:, 9] = False
    assert (got[clean] - plain[0, 0][clean]).norm() <= 1e-6 * plain.norm()
