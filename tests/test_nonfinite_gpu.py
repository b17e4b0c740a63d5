"""KQKV with a non-finite live value (a q value beyond f16's range, a NaN in a live cache row): the tokens
and heads it belongs to come out non-finite, whichever kernels the token and split counts pick, and the
others keep their bits."""
import math

import pytest
import torch

import aubier_amd as A
from oracle import oracle as orc

pytestmark = pytest.mark.gpu

N_KV, H = 2048, 96                               # 96 heads: every merge kernel is reached


def inputs(nt, dk, cache, dev):
    """The last token sees the whole window, the others its first half (or none of the last split)."""
    g = torch.Generator().manual_seed(nt)
    kc = torch.randn((N_KV, dk), generator=g)
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    mask = torch.zeros((nt, N_KV))
    mask[:-1, N_KV // 2:] = -math.inf
    if cache == "q8":
        kc = torch.from_numpy(orc.q8_0_quantize(kc.half().float().numpy()))
    else:
        kc = kc.half()
    return kc, q, mask.to(dev)


def kqkv(kc, dk, q, mask, split, dv, dev):
    kc = A.Q8_0(kc.to(dev), dk) if kc.dtype == torch.uint8 else kc.to(dev)
    if split is None:
        return A.ggml_m4_kqkv(kc, q, mask, 0.07)
    part = A.ggml_m4_kqkv_partial(kc, q, mask, 0.07, split, d_v=dv)
    return A.ggml_m4_phase_merge(part, n_head=H, d_v=dv)


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("cache", ["f16", "q8"])
@pytest.mark.parametrize("nt", [1, 2, 4, 15, 16])
@pytest.mark.parametrize("split", [None, 5, 32])
def test_nonfinite_stays(dev, dk, dv, cache, nt, split):
    kc, q, mask = inputs(nt, dk, cache, dev)
    clean = kqkv(kc, dk, q, mask, split, dv, dev)
    assert torch.isfinite(clean).all()

    q_inf = q.clone()
    q_inf[nt - 1, 7, 3] = 1e5                    # inf as f16
    out = kqkv(kc, dk, q_inf, mask, split, dv, dev)
    assert not torch.isfinite(out[7, nt - 1]).any()
    out[7, nt - 1] = clean[7, nt - 1]
    assert torch.equal(out, clean)

    kc_nan = kc.clone()
    if cache == "q8":                            # the scale of the block that holds the first rope values
        kc_nan[N_KV - 5, dv // 32 * 34:dv // 32 * 34 + 2] = torch.tensor([0x00, 0x7e], dtype=torch.uint8)
    else:
        kc_nan[N_KV - 5, dv] = math.nan
    out = kqkv(kc_nan, dk, q, mask, split, dv, dev)
    assert not torch.isfinite(out[:, nt - 1]).any()          # V is finite: only the score is NaN
    assert torch.equal(out[:, :nt - 1], clean[:, :nt - 1])
