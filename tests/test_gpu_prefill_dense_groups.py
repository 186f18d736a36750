"""The dense prefill's workgroup shapes (128 tokens x 1 key group, 64 x 2, 32 x 4):
lengths that leave key groups without a block, ragged windows and blocks, and
the sizes where the shape changes, against the float64 oracle; and the exact
walk of every group after a score far above block 0's."""

import numpy as np
import pytest
import torch

import sparda
from sparda import synth
from oracle import sparda_oracle as O
from helpers import assert_close_out, np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("R", [1, 3, 4])
@pytest.mark.parametrize("B,T,causal", [
    (1, 31, True), (1, 64, False), (1, 65, True),           # one block; two
    (1, 193, True), (2, 321, False), (16, 100, True),       # four groups
    (17, 193, True), (16, 250, False), (1, 5121, True),     # two
    (43, 130, True), (33, 129, False), (65, 65, True)])     # more windows than CUs: one
def test_dense_prefill_key_groups(R, B, T, causal):
    print(f"[case] dense groups R={R} B={B} T={T} causal={causal}", flush=True)
    x = synth.prefill_inputs(B, T, 4 * R, 4, 64, dtype=torch.bfloat16, seed=700 + T)
    out = sparda.prefill(x["q"].to(DEV), x["k"].to(DEV), x["v"].to(DEV), None, None, 64, causal=causal)
    r = np.random.default_rng(T)
    rows = sorted({(b, int(t)) for b in range(B) for t in r.integers(0, T, 16)} | {(0, 0), (B - 1, T - 1)})
    want = O.attention_prefill(np32(x["q"]), np32(x["k"]), np32(x["v"]), None, None, 64, causal, rows=rows)
    mask = np.zeros(want.shape, bool)
    for b, t in rows:
        mask[b, t] = True
    assert_close_out(np32(out), want, torch.bfloat16, mask)


@pytest.mark.parametrize("B,hot_key", [(1, 70), (1, 130), (1, 200), (1, 260),  # a block of each of four key groups
                                       (6, 70), (6, 260), (14, 260)])         # of two, of one
def test_dense_prefill_exact_walk_over_every_key_group(B, hot_key):
    print(f"[case] dense exact walk, B={B} hot key {hot_key}", flush=True)
    x = synth.prefill_inputs(B, 320, 12, 4, 64, dtype=torch.float32, seed=95)
    q, k, v = x["q"].clone(), x["k"].clone(), x["v"].clone()
    e = torch.zeros(64)
    e[0] = 20.0
    q[0, 300], k[0, 300], k[0, 0], k[0, hot_key] = e, -e, -e, e  # 72 log2-units above the other scores
    q, k, v = (t.to(torch.bfloat16) for t in (q, k, v))
    out = np32(sparda.prefill(q.to(DEV), k.to(DEV), v.to(DEV), None, None, 64))
    assert_close_out(out[:1], O.attention_prefill(np32(q[:1]), np32(k[:1]), np32(v[:1]), None, None, 64, True),
                     torch.bfloat16)
