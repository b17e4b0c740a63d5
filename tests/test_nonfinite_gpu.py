"""KQKV with a non-finite live value (a q value that is NaN or beyond its range, NaN in one live cache row or in
every one of a split): the tokens and heads it belongs to come out non-finite, whichever kernels the token
and split counts pick, and the others keep their bits.  Cells that no token sees may hold NaN."""
import math

import pytest
import torch

import aubier_amd as A
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

N_KV, H = 2048, 96                               # 96 heads: every merge kernel is reached
HOLE = slice(1280, 1344)                         # a tile that no token sees; a split of its own with 32 splits


def inputs(nt, dk, cache, dev):
    """The last token sees the whole window, the others its first half (or none of the last split)."""
    g = torch.Generator().manual_seed(nt)
    kc = torch.randn((N_KV, dk), generator=g)
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    mask = torch.zeros((nt, N_KV))
    mask[:-1, N_KV // 2:] = -math.inf
    mask[:, HOLE] = -math.inf
    if cache == "q8":
        kc = torch.from_numpy(orc.q8_0_quantize(kc.half().float().numpy()))
    elif cache == "f16":
        kc = kc.half()
    return kc, q, mask.to(dev)


def kqkv(kc, dk, q, mask, split, dv, dev):
    kc = A.Q8_0(kc.to(dev), dk) if kc.dtype == torch.uint8 else kc.to(dev)
    if split is None:
        return A.ggml_m4_kqkv(kc, q, mask, 0.07, out=torch.empty((H, q.shape[0], dv), device=dev))
    part = A.ggml_m4_kqkv_partial(kc, q, mask, 0.07, split, d_v=dv)
    return A.ggml_m4_phase_merge(part, n_head=H, d_v=dv)


def with_nan(kc, rows, dv):
    """NaN among the rows' rope values (the scale of the block that holds the first), so that V stays finite."""
    kc = kc.clone()
    if kc.dtype == torch.uint8:
        kc[rows, dv // 32 * 34:dv // 32 * 34 + 2] = torch.tensor([0x00, 0x7e], dtype=torch.uint8)
    else:
        kc[rows, dv] = math.nan
    return kc


# (192, 128): the VALU kernel, in splits that the other tokens do not see (in their own a NaN cell counts)
CASES = [(dk, dv, c, s) for dk, dv in ((576, 512), (320, 256)) for c in ("f16", "q8", "f32") for s in (None, 5, 32)]


@pytest.mark.parametrize("dk,dv,cache,split", CASES + [(192, 128, "f16", 32), (192, 128, "f32", 32)])
@pytest.mark.parametrize("nt", [1, 2, 4, 15, 16])
def test_nonfinite_stays(dev, dk, dv, cache, split, nt):
    kc, q, mask = inputs(nt, dk, cache, dev)
    clean = kqkv(kc, dk, q, mask, split, dv, dev)
    assert torch.isfinite(clean).all()

    for bad in (math.inf if cache == "f32" else 1e5, math.nan):          # 1e5: inf as f16
        q_bad = q.clone()
        q_bad[nt - 1, 7, 3] = bad
        out = kqkv(kc, dk, q_bad, mask, split, dv, dev)
        assert not torch.isfinite(out[7, nt - 1]).any(), bad
        out[7, nt - 1] = clean[7, nt - 1]
        assert torch.equal(out, clean), bad

    for rows in (slice(N_KV - 5, N_KV - 4), slice(N_KV - 64, N_KV)):
        out = kqkv(with_nan(kc, rows, dv), dk, q, mask, split, dv, dev)
        assert not torch.isfinite(out[:, nt - 1]).any(), rows
        assert torch.equal(out[:, :nt - 1], clean[:, :nt - 1]), rows

    if split == 32:
        assert torch.equal(kqkv(with_nan(kc, HOLE, dv), dk, q, mask, split, dv, dev), clean)
