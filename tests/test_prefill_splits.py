"""CPU test of the prefill split rule, read off the workspace it asks for: never more splits than one
workgroup per CU and split unit gives (so a workspace that was large enough stays so), and a count
whose time is near the best one's, by times measured on the MI355X over every count."""
import pytest
import torch

import aubier_amd as A
from aubier_amd import ops


def splits(n_kv, nt, H, dk, dv):
    kc, q, out = torch.zeros((n_kv, dk), dtype=torch.float16), torch.zeros((nt, H, dk)), torch.zeros((H, nt, dv))
    need = A.kqkv_workspace_bytes(kc, q, out)
    per = (H + 31) // 32 * nt * ops.part_floats(dv) * 4
    assert need % per == 0
    return max(1, need // per)


@pytest.mark.parametrize("dk,dv", [(576, 512), (320, 256)])
@pytest.mark.parametrize("H", [1, 32, 33, 128])
@pytest.mark.parametrize("nt", [16, 17, 63, 64, 250, 257, 500, 1000, 1030])
def test_prefill_split_range(dk, dv, H, nt):
    groups = (H + 31) // 32 * ((nt + 3) // 4)
    for n_kv in (1, 64, 65, 256, 1000, 2048, 8192, 40000):
        tiles = (n_kv + 63) // 64
        assert 1 <= splits(n_kv, nt, H, dk, dv) <= min(tiles, -(-256 // groups))


# us of KQKV (32 heads, the last nt keys causal) at 1, 2, ... splits, to the largest count of the range above
MEASURED = {
    (576, 64, 164): (29.7, 26.4, 25.5),
    (576, 152, 252): (35.1, 30.9, 30.0, 29.7),
    (576, 192, 292): (38.0, 33.4, 31.2, 33.6, 32.3),
    (576, 192, 1216): (79.0, 53.9, 46.9, 44.7, 43.9, 66.7),
    (576, 320, 420): (43.8, 39.3, 37.4, 58.1),
    (576, 400, 1000): (70.6, 54.6, 72.1),
    (576, 400, 500): (47.0, 41.3, 40.7),
    (576, 512, 4608): (235.7, 149.9),
    (576, 640, 740): (58.5, 75.7),
    (576, 1000, 1000): (74.3, 106.6),
    (320, 192, 1216): (53.1, 37.1, 31.8, 29.4, 28.9, 44.2),
    (320, 192, 292): (24.4, 22.5, 22.4, 22.4, 21.6),
    (320, 320, 420): (29.3, 26.5, 25.2, 38.3),
    (320, 512, 612): (35.7, 31.6),
    (320, 1000, 1000): (50.0, 68.1),
}


@pytest.mark.parametrize("dk,nt,n_kv", MEASURED)
def test_prefill_split_choice(dk, nt, n_kv):
    us = MEASURED[dk, nt, n_kv]
    assert us[splits(n_kv, nt, 32, dk, {576: 512, 320: 256}[dk]) - 1] <= 1.05 * min(us)


@pytest.mark.parametrize("dk,dv,H,nt,n_kv", [(576, 512, 32, 256, 256), (576, 512, 32, 512, 512), (576, 512, 32, 512, 612),
                                             (576, 512, 1, 60, 2000), (576, 512, 32, 340, 340), (576, 512, 128, 128, 200)])
def test_short_chunks_fit_the_no_alloc_array(dk, dv, H, nt, n_kv):
    """Counts whose records pass the array by little are given up where they gain little."""
    per = (H + 31) // 32 * nt * ops.part_floats(dv) * 4
    sp = splits(n_kv, nt, H, dk, dv)
    assert sp == 1 or sp * per <= ops.NOALLOC_SCRATCH_BYTES
