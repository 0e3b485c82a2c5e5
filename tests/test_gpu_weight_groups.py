"""The native backward with the weight gradients of several blocks in one launch against the single calls: one step of the
contraction and many (whole ones: token counts are multiples of 64), tiles that end inside in both directions, two groups of unequal size, and
gradients off the 16-byte grid, which are formed block by block."""
import ctypes

import pytest
import torch

from oracle import gpt2 as ogpt2
from util import DTYPES

pytestmark = pytest.mark.gpu
DEV = "cuda"


def both(mt, lo, monkeypatch, dtype, D, F, L, B, T, shift=0):
    V, H = 101, D // 64
    params = [[p.to(DEV).to(dtype) for p in grp] for grp in ogpt2.init_transformer_gpt2(V, D, L, H, F, T, seed=3)]
    y = torch.randint(0, V, (B, T + 1), generator=torch.Generator().manual_seed(7)).to(DEV)
    empty_like = torch.empty_like
    if shift:
        def off_the_grid(p, **kw):
            if tuple(p.shape) not in ((D, D), (F, D), (D, F), (H, 3, 64, D)):
                return empty_like(p, **kw)
            return torch.empty(p.numel() + shift, dtype=p.dtype, device=p.device)[shift:].view(p.shape)
        monkeypatch.setattr(mt.torch, "empty_like", off_the_grid)
    runs = []
    for native in (True, False):
        monkeypatch.setattr(mt, "NATIVE_STACK", native)
        grads, _ = lo.t_loss_bkwd3_t(params, y, None, None, True, list(range(10, 11 + 3 * L)))
        runs.append([p for grp in grads for p in grp])
    return runs


@pytest.mark.parametrize("dtype", DTYPES)
@pytest.mark.parametrize("D,F,L,B,T,shift", [(768, 3072, 2, 1, 64, 0), (768, 3072, 3, 3, 192, 0), (320, 1288, 17, 1, 320, 0),
                                             (768, 3080, 2, 1, 448, 0), (768, 3072, 2, 1, 128, 1), (256, 1024, 12, 7, 64, 0)])
def test_weight_gradients_together(mt, lo, monkeypatch, dtype, D, F, L, B, T, shift):
    runs = both(mt, lo, monkeypatch, dtype, D, F, L, B, T, shift)
    # The sums of a weight gradient are added in another order: in fp32 a few roundings of 2^-24; in bf16 a value on the edge may be
    # stored one step of 2^-8 away, all of them two independent roundings of 2^-9 / sqrt(3) at the very most.  Everything else
    # comes from the same products; of the pairs' (shift) in bf16 up to six stored tensors lie between two products of a block.
    bound = 2e-6 if dtype == torch.float32 else 1.6e-3 * (L * 6 if shift else 1) ** 0.5
    for i, (a, b) in enumerate(zip(*runs)):
        a, b = a.double(), b.double()
        assert (a - b).norm() <= bound * b.norm(), i


@pytest.mark.parametrize("dtype", DTYPES)
def test_workspace_of_one_block(mt, lo, monkeypatch, dtype):
    """A workspace without room for what several blocks' weight gradients read: the blocks one by one, in nothing but that room."""
    L, B, T, D, F, H = 3, 1, 64, 768, 3072, 12
    params = [[p.to(DEV).to(dtype) for p in grp] for grp in ogpt2.init_transformer_gpt2(101, D, L, H, F, T, seed=3)]
    flat = mt._native_params(params)
    y = torch.randint(0, 101, (B, T), generator=torch.Generator().manual_seed(7)).to(DEV)
    h, x_last, acts = mt._native_fwd(params, flat, y, None, True, list(range(10, 11 + 3 * L)), True)
    dh = torch.randn(h.shape, generator=torch.Generator().manual_seed(8)).to(DEV).to(dtype)
    lib = mt.lib()
    row = B * T * D * (2 if dtype == torch.bfloat16 else 4)
    whole = lib.ptj_gpt2_workspace_bytes(acts.shape, 1)
    # two blocks' d(feed-forward), d(qkv), d(residual) and one more entering gradient
    small = whole - 2 * (F // D + 3 + 1) * row - row

    def backward(ws_bytes, room):
        grads = [torch.zeros_like(p) for p in flat]
        demb = torch.empty_like(dh)
        ws = torch.full((room + 4096,), 7, dtype=torch.uint8, device=DEV)
        rc = lib.ptj_gpt2_bwd(acts.shape, mt._pointers(flat), None, acts.seeds, acts.buf.data_ptr(), acts.buf.numel(), x_last.data_ptr(),
                              dh.data_ptr(), mt._pointers(grads), demb.data_ptr(), ws.data_ptr(), ws_bytes, mt.stream())
        assert bool((ws[room:] == 7).all())
        return rc, [g.double() for g in grads[3:]] + [demb.double()]

    rc, want = backward(whole, whole)
    assert rc == 0
    rc, got = backward(small, small)
    assert rc == 0
    # as above; in bf16 up to six stored tensors lie between two products of a block
    bound = 2e-6 if dtype == torch.float32 else 1.6e-3 * (L * 6) ** 0.5
    for i, (a, b) in enumerate(zip(got, want)):
        assert (a - b).norm() <= bound * b.norm(), i
    assert backward(small - 1, small)[0] != 0


def test_out_of_memory_takes_the_small_workspace(mt, lo, monkeypatch):
    """Where the room for several blocks' weight gradients is not to be had, a step runs in that for one block; where that is not to be had
    either, the error is torch's."""
    L, T, D, F, H = 3, 64, 768, 3072, 12
    params = [[p.to(DEV) for p in grp] for grp in ogpt2.init_transformer_gpt2(101, D, L, H, F, T, seed=3)]
    y = torch.randint(0, 101, (1, T + 1), generator=torch.Generator().manual_seed(7)).to(DEV)
    seeds = list(range(10, 11 + 3 * L))
    want, _ = lo.t_loss_bkwd3_t(params, y, None, None, True, seeds)
    shape = (ctypes.c_int64 * 9)(L, 1, T, D, H, F, 101, 0, 1)
    whole, least = (mt.lib().ptj_gpt2_workspace_bytes(shape, b) for b in (1, 2))
    assert least < whole
    empty, asked = torch.empty, []

    def limited(limit):
        def f(*args, **kw):
            if args and args[0] in (whole, least):
                asked.append(args[0])
                if args[0] > limit:
                    raise torch.OutOfMemoryError("no room")
            return empty(*args, **kw)
        return f

    monkeypatch.setattr(mt.torch, "empty", limited(least))
    got, _ = lo.t_loss_bkwd3_t(params, y, None, None, True, seeds)
    assert asked == [whole, least]
    for a, b in zip([p for g in got for p in g], [p for g in want for p in g]):
        assert (a.double() - b.double()).norm() <= 2e-6 * b.double().norm()
    monkeypatch.setattr(mt.torch, "empty", limited(least - 1))
    with pytest.raises(torch.OutOfMemoryError):
        lo.t_loss_bkwd3_t(params, y, None, None, True, seeds)
