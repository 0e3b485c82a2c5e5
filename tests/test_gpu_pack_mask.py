"""The bit-packed attention mask: words in both orientations and tile classes against their definition (include/ptj.h), with an odd
number of tiles, masks that start at any byte, and bytes other than 0 and 1."""
import importlib

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def packed_by_definition(m):
    B, T, _ = m.shape
    G = T // 32
    bit = (np.uint64(1) << np.arange(32, dtype=np.uint64))
    by_key = (m.reshape(B, G, 32, T).astype(np.uint64) * bit[None, None, :, None]).sum(2)                # [B, G, T]
    by_query = (m.reshape(B, T, G, 32).astype(np.uint64) * bit).sum(3).transpose(0, 2, 1)                # [B, G, T]
    causal = np.tril(np.ones((T, T), bool))
    eff = (m & causal).reshape(B, G, 32, G, 32)
    same = (eff == causal.reshape(G, 32, G, 32)[None]).all((2, 4))
    cls = np.where(same, 2, np.where(eff.any((2, 4)), 1, 0))                                              # [B, G(q), G(k)]
    return np.concatenate([x.reshape(-1).astype(np.uint32) for x in (by_key, by_query, cls, cls.transpose(0, 2, 1))])


@pytest.mark.parametrize("B,T", [(1, 32), (3, 96), (2, 544), (5, 64)])
@pytest.mark.parametrize("shift", [0, 1, 7])
@pytest.mark.parametrize("kind", ["random", "causal", "packed", "none"])
def test_packed_words_and_classes(B, T, shift, kind):
    lib = importlib.import_module("pre-tjax_amd")._lib
    rng = np.random.default_rng(T + shift)
    m = np.tril(np.ones((T, T), bool))[None].repeat(B, 0)
    if kind == "random":
        m = rng.random((B, T, T)) < 0.5
    elif kind == "packed":
        doc = np.cumsum(rng.random((B, T)) < 4.0 / T, 1)
        m = m & (doc[:, :, None] == doc[:, None, :])
    elif kind == "none":
        m = np.zeros_like(m)
    raw = np.where(m, rng.integers(1, 256, m.shape), 0).astype(np.uint8) if kind == "random" else m.astype(np.uint8)
    buf = torch.full((shift + raw.size,), 1, dtype=torch.uint8, device="cuda")
    buf[shift:] = torch.from_numpy(raw.reshape(-1)).cuda()
    words = lib.lib().ptj_attn_packed_mask_bytes(B, T) // 4
    out = torch.full((words + 4,), -7, dtype=torch.int32, device="cuda")
    lib.check(lib.lib().ptj_attn_pack_mask(buf.data_ptr() + shift, out.data_ptr(), B, T, lib.stream()), "pack")
    got = out.cpu().numpy()
    assert (got[words:] == -7).all()
    assert np.array_equal(got[:words].view(np.uint32), packed_by_definition(m))
