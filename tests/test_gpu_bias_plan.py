"""A product with a bias and nothing behind it runs its own second stage of a K split, so it is planned as one without a bias is; the
second product of a block, whose partial sums the next norm adds up, may be split otherwise, in the native stack and call by call."""
import pytest
import torch

from oracle import gpt2 as ogpt2
from util import gen, randn

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("rows", [64, 300, 700, 750, 812, 1399, 1450, 1536, 3001, 9000])
def test_bias_does_not_change_the_plan(mt, rows):
    """Another split adds in another order, which some of the stored values show."""
    g = gen(rows)
    x, w = randn(g, rows, 3072).to(DEV).bfloat16(), randn(g, 768, 3072).to(DEV).bfloat16()
    zero = torch.zeros(768, dtype=torch.bfloat16, device=DEV)
    assert torch.equal(mt.matmul_t(x, w.t(), zero), mt.matmul_t(x, w.t()))


@pytest.mark.parametrize("B,T", [(11, 64), (23, 64), (2, 256)])
def test_native_stack_where_the_plans_differ(mt, monkeypatch, B, T):
    params = [[p.to(DEV).bfloat16() for p in grp] for grp in ogpt2.init_transformer_gpt2(101, 768, 2, 12, 3072, T, seed=3)]
    y = torch.randint(0, 101, (B, T), generator=torch.Generator().manual_seed(6)).to(DEV)
    runs = []
    for native in (True, False):
        monkeypatch.setattr(mt, "NATIVE_STACK", native)
        runs.append(mt.t_gpt2_forward_t(params, y, None, None, True, list(range(10, 17))))
    assert torch.equal(*runs)
