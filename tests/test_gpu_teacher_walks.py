"""The teacher block mass over its workgroup shapes and walks: window edges,
more blocks than a window keeps (row sums first, block sums in parts), and
scores far above those before (the reference raised, once and many times, and
after a block of -inf scores). fp32 sums of at most T terms: 1e-6 per
probability against float64. Infinite and NaN elements stay with their own rows."""

import numpy as np
import pytest
import torch

import sparda
from oracle import sparda_oracle as O
from helpers import np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,T,Hq,Hkv,causal,hot", [
    (1, 31, 12, 4, True, False), (1, 33, 8, 4, False, False), (1, 64, 4, 4, True, False),
    (33, 250, 12, 4, True, False),            # 64-token windows, ragged
    (1, 4161, 3, 1, True, False), (1, 4161, 1, 1, False, False),  # 66 blocks: written in parts
    (1, 300, 12, 4, True, True), (1, 4161, 3, 1, True, True)])
def test_teacher_mass_shapes(B, T, Hq, Hkv, causal, hot):
    print(f"[case] teacher walks B={B} T={T} Hq={Hq} Hkv={Hkv} causal={causal} hot={hot}", flush=True)
    g = torch.Generator().manual_seed(T + Hq)
    q = torch.randn(B, T, Hq, 64, generator=g)
    k = torch.randn(B, T, Hkv, 64, generator=g)
    if hot:
        q[0, T - 20], k[0, T - 90] = 1.5, 3.0  # 288 / 8 = 52 log2-units above a zero score
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    got = sparda.teacher_block_mass(q.to(DEV), k.to(DEV), 64, causal=causal).cpu().numpy()
    want = O.teacher_block_mass(np32(q[-1:]), np32(k[-1:]), 64, causal)
    assert np.abs(got[-1:] - want).max() < 1e-6 * (4 if hot else 1)
    assert np.abs(got.sum(-1) - 1.0).max() < 1e-5


@pytest.mark.parametrize("T,Hq,Hkv", [(500, 12, 4), (500, 4, 4), (4200, 2, 1)])
def test_teacher_mass_rising_scores(T, Hq, Hkv):
    # every row's scores rise by 24 log2-units from block to block of its last few: each raises the reference
    print(f"[case] teacher rising T={T} Hq={Hq} Hkv={Hkv}", flush=True)
    g = torch.Generator().manual_seed(T)
    q, k = torch.randn(1, T, Hq, 64, generator=g), torch.randn(1, T, Hkv, 64, generator=g)
    b = torch.arange(T) // 64
    q[..., 0] = 8.0
    k[..., 0] = (16.0 * torch.clamp(b - (T // 64 - 5), min=0)).to(torch.float32)[None, :, None]
    k[:, :64, :, 0] = float("-inf")  # block 0: nothing
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    got = sparda.teacher_block_mass(q.to(DEV), k.to(DEV), 64).cpu().numpy()
    want = O.teacher_block_mass(np32(q), np32(k), 64, True)
    assert np.abs(got[:, :, 64:] - want[:, :, 64:]).max() < 4e-6
    assert np.isnan(got[:, :, :64, 0]).all()  # rows with no finite score


@pytest.mark.parametrize("R", [1, 2, 3])
@pytest.mark.parametrize("bad", [float("nan"), float("inf"), float("-inf")])
def test_teacher_mass_bad_elements_stay_in_their_rows(R, bad):
    print(f"[case] teacher R={R} element {bad}", flush=True)
    T, row, key = 200, 37, 150
    g = torch.Generator().manual_seed(9)
    q, k = torch.randn(1, T, R, 64, generator=g), torch.randn(1, T, 1, 64, generator=g)
    q, k = q.to(torch.bfloat16), k.to(torch.bfloat16)
    want = sparda.teacher_block_mass(q.to(DEV), k.to(DEV), 64).cpu().numpy()
    q[0, row, 0, 5], k[0, key, 0, 7] = bad, bad
    got = sparda.teacher_block_mass(q.to(DEV), k.to(DEV), 64).cpu().numpy()
    clean = [t for t in range(key) if t != row]  # rows before the key, but the one
    assert np.abs(got[:, :, clean] - want[:, :, clean]).max() < 1e-6
    assert np.isnan(got[0, 0, row]).any()
