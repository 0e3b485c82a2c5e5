"""CPU-only: a null entry in the parameter or gradient nest of the native stack is refused before anything is launched, whichever way
the products of its size are launched."""
import ctypes
import importlib

import pytest
import torch

# GPU addresses that nothing may read: on the CPU a call that is not refused fails in its first launch
pytestmark = pytest.mark.skipif(torch.cuda.is_available(), reason="calls with made-up addresses")
FIRST, BLOCK = 3, 10                       # include/ptj.h: ptj_gpt2_fwd
LN1G, LN1B, WQKV, WO, LN2G, LN2B, W1, B1, W2, B2 = range(BLOCK)


def nest(layers, missing=None):
    entries = [0x1000 * (i + 1) for i in range(FIRST + BLOCK * layers + 2)]
    if missing is not None:
        entries[missing] = None
    return (ctypes.c_void_p * len(entries))(*entries)


def shape(layers, tokens, dtype):
    return (ctypes.c_int64 * 9)(layers, 1, tokens, 768, 12, 3072, 101, dtype, 0)


def backward(layers, tokens, dtype, missing_grad=None, missing_param=None):
    l = importlib.import_module("pre-tjax_amd._lib").lib()
    big = 1 << 50
    rc = l.ptj_gpt2_bwd(shape(layers, tokens, dtype), nest(layers, missing_param), None, None, 0x100000, big, 0x200000, 0x300000,
                        nest(layers, missing_grad), 0x400000, 0x500000, big, None)
    return rc, l.ptj_last_error()


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("layers,tokens", [(1, 64), (2, 64), (12, 4096)])       # block by block and in groups
@pytest.mark.parametrize("which", [WQKV, WO, W1, B1, W2])
def test_backward_refuses_missing_weight_gradients(dtype, layers, tokens, which):
    for block in (0, layers - 1):
        rc, message = backward(layers, tokens, dtype, missing_grad=FIRST + BLOCK * block + which)
        assert rc == -1 and b"null" in message


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("which", [LN1G, WQKV, WO, LN2G, W1, W2])
def test_backward_refuses_missing_weights(dtype, which):
    rc, message = backward(2, 64, dtype, missing_param=FIRST + BLOCK + which)
    assert rc == -1 and b"null" in message


def forward(layers, tokens, dtype, keep, missing):
    l = importlib.import_module("pre-tjax_amd._lib").lib()
    big = 1 << 50
    rc = l.ptj_gpt2_fwd(shape(layers, tokens, dtype), nest(layers, missing), 0x600000, None, None, 0x100000, big, keep, 0x200000,
                        0x300000, 0x500000, big, None)
    return rc, l.ptj_last_error()


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("keep", [0, 1])
@pytest.mark.parametrize("tokens", [64, 4096])                 # bf16: each norm inside the product that reads it, or apart
@pytest.mark.parametrize("which", [LN1G, LN1B, WQKV, WO, LN2G, LN2B, W1, B1, W2])
def test_forward_refuses_missing_parameters(dtype, keep, tokens, which):
    for block in (0, 1):
        rc, message = forward(2, tokens, dtype, keep, FIRST + BLOCK * block + which)
        assert rc == -1 and b"null" in message


@pytest.mark.parametrize("entry", [0, 1])
def test_forward_refuses_a_missing_final_norm(entry):
    rc, message = forward(2, 64, 1, 0, FIRST + BLOCK * 2 + entry)
    assert rc == -1 and b"null" in message
