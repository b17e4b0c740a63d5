"""Rows (tokens) of a decode call that share a split's workgroup: four live rows at a time through the
prefill pass, fewer in turn.  Against float64 (the reference and the bar of the prefill tests), with
splits of at most one tile, and of three tiles with every row of a split in one workgroup (256
workgroups or more per row), where passes and single rows follow one another on one LDS ring; with splits
in which some rows have no live key, or in some tiles only, and empty splits.  (2500 keys in 13
splits: ten row groups, at most two rows each.)"""
import math

import pytest
import torch

import aubier_amd as A

from test_prefill_live_gpu import check, reference

pytestmark = pytest.mark.gpu


def masks(kind, nt, n_kv, g):
    m = torch.full((nt, n_kv), -math.inf)
    for t in range(nt):
        if kind == "tail":                                   # drafted tokens at the end of one window
            m[t, :n_kv - nt + t + 1] = 0.0
        elif kind == "regions":                              # sequences of their own, some overlapping
            a = (t * n_kv) // nt
            m[t, a:a + 1 + (n_kv // nt) * (1 + t % 3)] = 0.0
        elif kind == "tiles":                                # every third tile, another one for the next row
            for k in range(64 * (t % 3), n_kv, 192):
                m[t, k + t:k + 64] = 0.0
        else:                                                # some rows dead in some splits, one row dead
            m[t] = torch.where(torch.rand(n_kv, generator=g) < 0.02, 0.0, -math.inf)
            m[t, 64 * t:64 * t + 64] = -math.inf
            m[t, n_kv - 1] = 0.0
            if t == 1:
                m[t] = -math.inf
    return m


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("nt", [2, 3, 4, 5, 7, 8, 15])
@pytest.mark.parametrize("kind", ["none", "tail", "regions", "holes"])
@pytest.mark.parametrize("n_kv,split", [(1000, 256), (2500, 13), (130, 300)])
def test_shared_rows(dev, dk, dv, nt, kind, n_kv, split):
    run(dev, dk, dv, nt, kind, n_kv, split)


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("nt", [3, 5, 7, 8, 15])
@pytest.mark.parametrize("kind", ["none", "tail", "regions", "holes", "tiles"])
def test_splits_of_several_tiles(dev, dk, dv, nt, kind):
    run(dev, dk, dv, nt, kind, 128 * 64 * 3 + 17, 128)


def run(dev, dk, dv, nt, kind, n_kv, split):
    g = torch.Generator().manual_seed(n_kv + nt)
    H, scale = 40, 1.0 / math.sqrt(192.0)
    kc = torch.randn((n_kv, dk), generator=g).half().to(dev)
    q = torch.randn((nt, H, dk), generator=g).to(dev)
    mask = None if kind == "none" else masks(kind, nt, n_kv, g).to(dev)
    part = A.ggml_m4_kqkv_partial(kc, q, mask, scale, split, d_v=dv)
    ref = reference(kc, q, torch.zeros((nt, n_kv), device=dev) if mask is None else mask, scale, dv)
    check(f"{kind} nt={nt}", A.ggml_m4_phase_merge(part, n_head=H, d_v=dv), ref)


def test_rows_over_a_window_of_256_tiles(dev):
    g = torch.Generator().manual_seed(2)
    n_kv, nt, H = 16400, 4, 32
    kc = torch.randn((n_kv, 576), generator=g).half().to(dev)
    q = torch.randn((nt, H, 576), generator=g).to(dev)
    mask = masks("tail", nt, n_kv, g).to(dev)
    check("16,400 keys", A.ggml_m4_kqkv(kc, q, mask, 0.07), reference(kc, q, mask, 0.07, 512))
