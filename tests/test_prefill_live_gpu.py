"""Prefill KQKV over masks that leave each token a run of live keys of its own: the kernel's loop runs
over the tiles its workgroup's tokens see, found from the two ends of the mask rows.  Against float64
on the values the kernel computes with (q rounded to f16).  Bar: q and P each enter with an f16
rounding (2^-11 of a score's terms, 2^-11 of a weight), the records once more; 3e-3 of max |ref|, the
f16-cache bar of the other prefill tests."""
import math

import pytest
import torch

import aubier_amd as A

from conftest import say

pytestmark = pytest.mark.gpu

BAR = 3e-3


def reference(kc, q, mask, scale, dv):
    k, qd = kc.double(), q.half().double()
    out = torch.zeros((q.shape[1], q.shape[0], dv), dtype=torch.float64, device=q.device)
    live = (mask > -math.inf).any(dim=1)
    for h in range(q.shape[1]):
        s = (qd[:, h].contiguous() @ k.t().contiguous()) * scale + mask.double()
        out[h, live] = torch.softmax(s[live], dim=-1) @ k[:, :dv].contiguous()
    return out                                   # a token with no live key: 0


def check(name, out, ref):
    err = (out.double() - ref).abs().max().item() / ref.abs().max().item()
    say(f"{name}: {err:.2e} of max|ref|")
    assert torch.isfinite(out).all() and err <= BAR, (name, err)


def runs(kind, nt, n_kv, g):
    """[first, last) of each token's live keys."""
    r = []
    for t in range(nt):
        if kind == "causal":
            r.append((0, max(1, n_kv - nt + t + 1)))
        elif kind == "edges":                    # around the 1,024-key rounds and the 64-key tiles
            e = (0, 1, 63, 64, 65, 127, 1023, 1024, 1025, 1087, n_kv - 1)[t % 11] % n_kv
            r.append((e, min(n_kv, e + (1, 2, 64, 65, 1024, 1025)[t % 6])))
        elif kind == "some_dead":                # whole workgroups and single tokens without a live key
            a = int(torch.randint(0, n_kv, (1,), generator=g))
            r.append((0, 0) if t % 3 == 0 or 4 <= t < 8 else (a, n_kv))
        else:
            a, b = sorted(torch.randint(0, n_kv + 1, (2,), generator=g).tolist())
            r.append((a, b))
    return r


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("n_kv", [40, 65, 1088, 2500])
@pytest.mark.parametrize("kind", ["causal", "edges", "some_dead", "random"])
@pytest.mark.parametrize("split", [None, 1, 3])
def test_live_runs(dev, dk, dv, n_kv, kind, split):
    g = torch.Generator().manual_seed(n_kv + dk)
    nt, H, scale = 21, 33, 1.0 / math.sqrt(192.0)
    kc = torch.randn((n_kv, dk), generator=g).half().to(dev)
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    mask = torch.full((nt, n_kv), -math.inf)
    for t, (a, b) in enumerate(runs(kind, nt, n_kv, g)):
        mask[t, a:b] = 0.25 * torch.randn(b - a, generator=g)
    mask = mask.to(dev)
    if split is None:
        out = A.ggml_m4_kqkv(kc, q, mask, scale)
    else:
        part = A.ggml_m4_kqkv_partial(kc, q, mask, scale, split, d_v=dv)
        out = A.ggml_m4_phase_merge(part, n_head=H, d_v=dv)
    check(f"{kind} n_kv={n_kv} split={split}", out, reference(kc, q, mask, scale, dv))


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
def test_sharp_scores_move_the_reference(dev, dk, dv):
    """Scores that grow by more than 2^15 along the window (the lazily moved reference moves and the
    accumulators are rescaled, also after tiles of masked keys)."""
    g = torch.Generator().manual_seed(5)
    nt, H, n_kv = 18, 32, 700
    kc = torch.randn((n_kv, dk), generator=g)
    kc[:, dv:] = 0.0
    kc[:, dv] = torch.arange(n_kv) / 16.0        # the score's drift: 44 nats over the window
    q = 0.02 * torch.randn((nt, H, dk), generator=g)
    q[:, :, dv] = 1.0
    mask = torch.zeros((nt, n_kv))
    mask[3, :200] = -math.inf
    mask[5, 100:400] = -math.inf
    kc, q, mask = kc.half().to(dev), q.to(dev), mask.to(dev)
    check("drift", A.ggml_m4_kqkv(kc, q, mask, 1.0), reference(kc, q, mask, 1.0, dv))
