"""CPU-only: the backward's workspace keeps what the weight gradients of several blocks read for no more blocks than make the launch
faster: groups that fill their rounds of tiles as well as all blocks together would."""
import ctypes
import importlib

import pytest

D, F = 768, 3072


def workspace(layers, tokens, dtype, backward=1):
    shape = (ctypes.c_int64 * 9)(layers, tokens // 64, 64, D, D // 64, F, 101, dtype, 0)
    return importlib.import_module("pre-tjax_amd._lib").lib().ptj_gpt2_workspace_bytes(shape, backward)


@pytest.mark.parametrize("dtype,tokens,blocks", [(1, 16384, 7), (1, 65536, 7), (0, 4096, 4), (0, 32768, 4)])
def test_a_part_of_the_blocks_is_kept(dtype, tokens, blocks):
    """bf16: seven blocks are 2.95 rounds of 256x256 tiles and five 2.8 of 256x192, all twelve 5.1 and 6.75; fp32: twelve 20.25 of 128x128,
    four 6.75."""
    a_block = tokens * (F + 5 * D) * (4 if dtype == 0 else 2)          # d(feed-forward), d(qkv), d(residual), the gradient that enters
    sums = 4 * ((tokens + 31) // 32 * F + 2 * 512 * 3 * D)             # and the partial rows of its column sums, which stay for all
    # a block that is not kept adds its partial rows (and its share of alignment) alone
    assert workspace(12, tokens, dtype) - workspace(blocks, tokens, dtype) <= (12 - blocks) * (sums + 4096)
    assert workspace(blocks, tokens, dtype) - workspace(2, tokens, dtype) >= (blocks - 2) * a_block


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("tokens", [64, 512, 1984])
def test_all_blocks_of_few_tokens(dtype, tokens):
    """Further launches cost 2 to 20 % of them (us in csrc/gemm_group.hip), what is kept is at most 28 MB a block in bf16."""
    a_block = tokens * (F + 5 * D) * (4 if dtype == 0 else 2)
    assert workspace(12, tokens, dtype) - workspace(7, tokens, dtype) >= 5 * a_block


@pytest.mark.parametrize("dtype", [0, 1])
@pytest.mark.parametrize("layers", [1, 2, 3, 12, 17, 48])
@pytest.mark.parametrize("tokens", [64, 512, 4096, 16384])
def test_never_more_than_sixteen_blocks(dtype, layers, tokens):
    a_block = tokens * (F + 5 * D) * (4 if dtype == 0 else 2)
    sums = 4 * ((tokens + 31) // 32 * F + 2 * 512 * 3 * D) + 4096
    assert workspace(layers, tokens, dtype) - workspace(1, tokens, dtype) <= min(layers, 16) * a_block + layers * sums


@pytest.mark.parametrize("dtype", [0, 1])
def test_the_least_that_is_taken(dtype):
    a_block = 4096 * (F + 5 * D) * (4 if dtype == 0 else 2)
    least, whole = workspace(12, 4096, dtype, 2), workspace(12, 4096, dtype)
    assert least <= whole - 2 * a_block
    assert workspace(1, 4096, dtype, 2) == workspace(1, 4096, dtype)
