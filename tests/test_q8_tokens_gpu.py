"""The many-token kernels of the Q8_0 ops (WKB and PHASE wv_b): bit-identical to the
oracle at the edges of their tiles (32 tokens, 128 outputs, 32-column blocks), and to the one-token
kernels for activations at the ends of the float range."""
import numpy as np
import pytest
import torch

import aubier_amd as A
from oracle import oracle as orc

from conftest import say

pytestmark = pytest.mark.gpu


def q8_dev(blocks_np, lead_shape, ne0, dev):
    return A.Q8_0(torch.from_numpy(np.ascontiguousarray(blocks_np)).reshape(*lead_shape, ne0 // 32 * 34).to(dev), ne0)


def same_bits(got, ref):
    return np.array_equal(np.ascontiguousarray(got).view(np.uint32), np.ascontiguousarray(ref).view(np.uint32))


@pytest.mark.parametrize("nt", [7, 8, 31, 32, 33, 97])
@pytest.mark.parametrize("d_in,d_out,H", [(256, 128, 96), (512, 136, 48), (256, 33, 320), (512, 161, 8), (256, 1, 400)])
def test_wvb_tokens(dev, nt, d_in, d_out, H):
    w = orc.q8_0_random(8700 + d_in + d_out, H * d_out, d_in)
    x = np.random.default_rng(8701 + nt).standard_normal((H, nt, d_in)).astype(np.float32)
    x[:, nt // 2] = 0.0                                  # a token of zeros: amax = 0 in every block
    ref = orc.wvb_q8(w, d_in, d_out, H, np.ascontiguousarray(x.transpose(1, 0, 2))).transpose(1, 0, 2)
    # strided views: dword-aligned rows, padding in the output that must stay as it is
    xd = torch.zeros((H, nt, d_in + 3), device=dev)
    xd[:, :, :d_in] = torch.from_numpy(x).to(dev)
    out = torch.full((H, nt, d_out + 5), 7.0, device=dev)
    A.ggml_m4_phase_wvb(q8_dev(w, (H, d_out), d_in, dev), xd[:, :, :d_in], out=out[:, :, :d_out])
    got = out.cpu().numpy()
    say(f"wv_b nt={nt} d_in={d_in} d_out={d_out}: max|diff|={np.abs(got[:, :, :d_out] - ref).max():.3e}")
    assert same_bits(got[:, :, :d_out], ref)
    assert (got[:, :, d_out:] == 7.0).all()


@pytest.mark.parametrize("nt", [7, 8, 31, 32, 33, 97])
@pytest.mark.parametrize("d_n,d_v,H", [(64, 256, 256), (128, 512, 32), (64, 33, 240), (128, 160, 32), (64, 1, 224)])
def test_wkb_tokens(dev, nt, d_n, d_v, H):
    w = orc.q8_0_random(8800 + d_n + d_v, H * d_v, d_n)
    q = np.random.default_rng(8801 + nt).standard_normal((nt, H, d_n + 65)).astype(np.float32)
    q[nt // 2] = 0.0
    ref = orc.wkb_q8(w, d_n, d_v, H, np.ascontiguousarray(q[:, :, :d_n]))
    out = torch.full((nt, H, d_v + 3), 7.0, device=dev)
    A.ggml_m4_wkb(q8_dev(w, (H, d_v), d_n, dev), torch.from_numpy(q).to(dev)[:, :, :d_n], out=out[:, :, :d_v])
    got = out.cpu().numpy()
    say(f"WKB Q8_0 nt={nt} d_n={d_n} d_v={d_v}: max|diff|={np.abs(got[:, :, :d_v] - ref).max():.3e}")
    assert same_bits(got[:, :, :d_v], ref)
    assert (got[:, :, d_v:] == 7.0).all()


def extreme(shape, seed):
    """Ordinary values, with tokens of subnormals, of huge values (f16 scales that overflow to inf),
    and with an inf or a NaN in one block."""
    x = np.random.default_rng(seed).standard_normal(shape).astype(np.float32)
    x[1] *= 1e-42
    x[2] *= 1e9
    x[3, :, 5] = np.inf
    x[4, :, 7] = np.nan
    x[5] *= 1e-30
    return x


def test_tokens_agree_with_one_token_kernels(dev):
    H, nt = 32, 64
    for d_in in (256, 512):
        w = q8_dev(orc.q8_0_random(8900 + d_in, H * 128, d_in), (H, 128), d_in, dev)
        x = torch.from_numpy(np.ascontiguousarray(extreme((nt, H, d_in), 8901).transpose(1, 0, 2))).to(dev)
        many = A.ggml_m4_phase_wvb(w, x).cpu().numpy()
        one = np.concatenate([A.ggml_m4_phase_wvb(w, x[:, t:t + 1]).cpu().numpy() for t in range(nt)], axis=1)
        np.testing.assert_array_equal(many, one)
    for d_n, d_v in ((64, 256), (128, 512)):
        w = q8_dev(orc.q8_0_random(8950 + d_n, H * d_v, d_n), (H, d_v), d_n, dev)
        q = torch.from_numpy(extreme((nt, H, d_n), 8951)).to(dev)
        many = A.ggml_m4_wkb(w, q).cpu().numpy()
        one = np.concatenate([A.ggml_m4_wkb(w, q[t:t + 1]).cpu().numpy() for t in range(nt)], axis=0)
        np.testing.assert_array_equal(many, one)
