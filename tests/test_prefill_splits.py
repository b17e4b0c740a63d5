"""CPU test of the prefill split rule, read off the workspace it asks for: never more splits than one
workgroup per CU and split unit gives (so a workspace or scratch that was large enough stays so), one
split for short windows, and no second round of workgroups where one round has room for every key."""
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
def test_prefill_split_rule(dk, dv, H, nt):
    groups = (H + 31) // 32 * ((nt + 3) // 4)
    for n_kv in (1, 64, 65, 256, 1000, 2048, 8192, 40000):
        tiles = (n_kv + 63) // 64
        cap = min(tiles, -(-256 // groups))
        sp = splits(n_kv, nt, H, dk, dv)
        assert 1 <= sp <= cap
        if sp > 1:
            assert groups * sp <= 256 or groups * (sp - 1) > 128
