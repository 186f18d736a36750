"""The fused producer's tiles (64, 128 and 256 rows, 32- and 64-wide steps):
row counts at their edges and a width that is no multiple of 64, against fp32."""

import pytest
import torch

import sparda
from model.rope import rope_tables
from helpers import assert_close_out, np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,T,C,nq,f_dtype", [(1, 63, 768, 768, torch.bfloat16), (1, 65, 96, 256, torch.float32),
                                              (3, 1820, 128, 768, torch.bfloat16), (1, 5500, 160, 1024, torch.float32),
                                              (5, 2300, 64, 768, torch.bfloat16),
                                              (5, 2783, 64, 768, torch.bfloat16)])  # 2.1, 2.6 workgroups a CU
def test_produce_tile_edges(B, T, C, nq, f_dtype):
    print(f"[case] produce tiles B={B} T={T} C={C} nq={nq}", flush=True)
    g = torch.Generator().manual_seed(T)
    nkv, nf, eps = 256, 256, 1e-5
    x = torch.randn(B, T, C, generator=g).to(torch.bfloat16).to(DEV)
    w = (0.05 * torch.randn(nq + 2 * nkv + nf, C, generator=g)).to(torch.bfloat16).to(DEV)
    cos, sin = (t.to(DEV) for t in rope_tables(64, T + 7))
    got = sparda.produce(x, w, nq, nkv, nf, eps, cos, sin, pos0=7, f_dtype=f_dtype)
    xf = x.float()
    y = (xf * torch.rsqrt(xf.pow(2).mean(-1, keepdim=True) + eps)) @ w.float().t()
    c, s = cos[7:7 + T][None, :, None, :], sin[7:7 + T][None, :, None, :]

    def rot(t):
        a, b = t[..., :32], t[..., 32:]
        return torch.cat((a * c - b * s, b * c + a * s), dim=-1)

    heads = [t.reshape(B, T, -1, 64) for t in y.split([nq, nkv, nkv, nf], -1)]
    for o, ref, name in zip(got, (rot(heads[0]), rot(heads[1]), heads[2], heads[3]), "qkvf"):
        assert_close_out(np32(o), np32(ref), torch.bfloat16, what=f"produce {name}")
