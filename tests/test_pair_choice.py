"""How the native backward launches the two products of a linear layer: a choice on sizes alone, made on the host."""
import ctypes
import importlib

import pytest

from test_gpu_native_stack import PAIRS

LAYERS = ((1, 4, True), (4, 1, False), (1, 1, False), (3, 1, False))      # outputs and inputs in widths; dX multiplied


def choice(n, m, k, multiplied):
    first = ctypes.c_int(-1)
    config = importlib.import_module("pre-tjax_amd._lib").lib().ptj_linear_bwd_choice(n, m, k, int(multiplied), ctypes.byref(first))
    return config, bool(first.value)


def test_the_gpu_test_sees_every_pair_of_tiles():
    """Pairs of equal tiles of 128 x 128 (9), all four of 64 x 64 and 64 x 128 (1, 2, 4, 5), either product first."""
    seen = {choice(B * T, a * D, b * D, mul) + (mul,) for D, B, T in PAIRS for a, b, mul in LAYERS}
    for mul in (False, True):
        assert {c for c, _, m in seen if m == mul} >= {1, 2, 4, 5, 9}
    for config in (4, 5, 9):
        assert {first for c, first, _ in seen if c == config} == {False, True}


@pytest.mark.parametrize("n,m,k,multiplied", [(12288, 256, 1024, True), (8192, 1024, 256, False), (6000, 768, 256, False),
                                              (12288, 1024, 256, False), (8192, 320, 1280, True), (6000, 320, 1280, True)])
def test_long_chains_of_narrow_layers(n, m, k, multiplied):
    """dW's chain alone takes longer than both products one after the other (two launches 8 to 31 % faster)."""
    assert choice(n, m, k, multiplied)[0] == 0


def test_refuses_what_the_backward_does_not_take():
    assert choice(0, 64, 64, False)[0] < 0 and choice(1 << 20, 64, 64, False)[0] < 0
