"""WKB with an f32 weight for 1-17 tokens (the row-sum kernel, the all-tokens-at-once kernel and the
GEMM's first size) against float64: 1e-6 of max |ref| (f32 products and sums over at most 128 values;
measured 3e-7), at 16 columns, head counts that end inside a workgroup, dword-aligned output rows."""
import pytest
import torch

import aubier_amd as A

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nt", [1, 3, 4, 5, 6, 15, 16, 17])
@pytest.mark.parametrize("d_n,d_v,H", [(128, 512, 32), (64, 256, 32), (64, 16, 3), (128, 16, 1), (128, 48, 5), (64, 80, 7)])
def test_wkb_few_tokens(dev, nt, d_n, d_v, H):
    g = torch.Generator().manual_seed(nt + d_v)
    w = torch.randn((H, d_v, d_n), generator=g).to(dev)
    q = torch.randn((nt, H, d_n + 64), generator=g).to(dev)[:, :, :d_n]
    out = torch.full((nt, H, d_v + 5), 7.0, device=dev)
    A.ggml_m4_wkb(w, q, out=out[:, :, 1:1 + d_v])
    ref = torch.stack([q[:, h].double() @ w[h].double().t().contiguous() for h in range(H)], dim=1)
    err = (out[:, :, 1:1 + d_v].double() - ref).abs().max() / ref.abs().max()
    assert err <= 1e-6, err
    assert (out[:, :, 0] == 7.0).all() and (out[:, :, 1 + d_v:] == 7.0).all()
