"""KQKV over an f32 cache at the MLA geometries (the f32-MFMA kernel) against float64.  Bar: f32
products and sums over D_k and the window; 1e-5 of max |ref|, the f32-cache bar of the other tests
(measured: below 2e-6)."""
import math

import pytest
import torch

import aubier_amd as A

from conftest import say

pytestmark = pytest.mark.gpu

BAR = 1e-5


def reference(kc, q, mask, scale, dv):
    k, qd = kc.double(), q.double()
    out = torch.zeros((q.shape[1], q.shape[0], dv), dtype=torch.float64, device=q.device)
    m = torch.zeros((q.shape[0], kc.shape[0]), device=q.device) if mask is None else mask
    live = (m > -math.inf).any(dim=1)
    for h in range(q.shape[1]):
        s = (qd[:, h].contiguous() @ k.t().contiguous()) * scale + m.double()
        out[h, live] = torch.softmax(s[live], dim=-1) @ k[:, :dv].contiguous()
    return out                                   # a token with no live key: 0


def check(name, out, ref):
    err = (out.double() - ref).abs().max().item() / max(1e-30, ref.abs().max().item())
    say(f"{name}: {err:.2e} of max|ref|")
    assert torch.isfinite(out).all() and err <= BAR, (name, err)


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("n_kv", [1, 15, 17, 32, 33, 63, 520, 1000, 2049])
@pytest.mark.parametrize("H,nt", [(1, 600), (560, 1), (33, 17), (128, 5)])
@pytest.mark.parametrize("split", [None, 1, 2, 7])
def test_edges(dev, dk, dv, n_kv, H, nt, split):
    g = torch.Generator().manual_seed(1000 * n_kv + H)
    kc = torch.zeros((n_kv, dk + 4))             # padded rows, as a view
    kc[:, :dk] = torch.randn((n_kv, dk), generator=g)
    kc = kc.to(dev)[:, :dk]
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    mask = None
    if n_kv % 2:
        mask = 0.5 * torch.randn((nt, n_kv), generator=g)
        mask[torch.rand((nt, n_kv), generator=g) < 0.3] = -math.inf
        mask = mask.to(dev)
    scale = 1.0 / math.sqrt(192.0)
    if split is None:
        out = A.ggml_m4_kqkv(kc, q, mask, scale, out=torch.empty((H, nt, dv), device=dev))
    else:
        part = A.ggml_m4_kqkv_partial(kc, q, mask, scale, split, d_v=dv)
        out = A.ggml_m4_phase_merge(part, n_head=H, d_v=dv)
    check(f"n_kv={n_kv} H={H} nt={nt} split={split}", out, reference(kc, q, mask, scale, dv))


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("H", [200, 4])
@pytest.mark.parametrize("split", [1, 3, 40])
def test_dead_splits_and_neighbours(dev, dk, dv, H, split):
    """Runs of masked keys longer than a split, on the f32-MFMA kernel and (4 heads) the VALU kernel; with 40
    splits of 16 keys some that no token sees hold infinities, which must not reach the result."""
    g = torch.Generator().manual_seed(9)
    n_kv, nt = 640, 3
    kc = torch.randn((n_kv, dk), generator=g)
    mask = torch.zeros((nt, n_kv))
    mask[0, :] = -math.inf                       # no live key at all
    mask[1, :320] = -math.inf
    mask[2, 200:] = -math.inf
    mask[2, 5] = 30.0                            # sharp
    kc, mask = kc.to(dev), mask.to(dev)
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    ref = reference(kc, q, mask, 0.07, dv)
    if split == 40:
        kc[208:320] = math.inf
    part = A.ggml_m4_kqkv_partial(kc, q, mask, 0.07, split, d_v=dv)
    m, l, _ = A.ops.decode_partials(part, H, d_v=dv) if split > 1 else (None, None, None)
    if m is not None:
        assert (m[:, 0] == -math.inf).all() and (l[:, 0] == 0).all()
    check(f"split={split}", A.ggml_m4_phase_merge(part, n_head=H, d_v=dv), ref)


@pytest.mark.parametrize("n_kv,split", [(48, 3), (80, 5)])
def test_rows_of_other_splits_stay_out(dev, n_kv, split):
    """A 16-key split is half a tile: the rows after it belong to the next split, here infinities in a
    masked split, and enter neither its scores nor its output."""
    kc = torch.randn((n_kv, 576), generator=torch.Generator().manual_seed(3))
    kc[16:32] = math.inf
    mask = torch.zeros((1, n_kv))
    mask[0, 16:32] = -math.inf
    q = torch.randn((1, 300, 576), generator=torch.Generator().manual_seed(4)).to(dev)
    part = A.ggml_m4_kqkv_partial(kc.to(dev), q, mask.to(dev), 0.07, split)
    m, l, o = A.ops.decode_partials(part, 300)
    keep = [s for s in range(split) if s != 1]
    k2, m2 = torch.cat([kc[:16], kc[32:]]).to(dev), torch.cat([mask[:, :16], mask[:, 32:]], dim=1).to(dev)
    part2 = A.ggml_m4_kqkv_partial(k2, q, m2, 0.07, split - 1)
    m_, l_, o_ = A.ops.decode_partials(part2, 300)
    assert (m[:, :, keep] == m_).all() and (l[:, :, keep] == l_).all() and (o[:, :, keep] == o_).all()
