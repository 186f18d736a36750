"""Dense decode over its split counts: one split, two, a last split of one key,
and more splits than one round of the merge holds, against the float64 oracle;
and keys whose scores are all -inf, in part of a split and in whole ones."""

import numpy as np
import pytest
import torch

import sparda
from sparda import synth
from oracle import sparda_oracle as O
from helpers import assert_close_out, np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("B,S,Hq,Hkv", [(1, 256, 12, 4), (2, 257, 12, 4), (3, 1025, 4, 4), (1, 33000, 8, 2),
                                        (1, 70000, 16, 1)])
def test_decode_dense_split_counts(B, S, Hq, Hkv):
    print(f"[case] decode dense B={B} S={S} Hq={Hq}", flush=True)
    y = synth.decode_inputs(B, S, Hq, Hkv, 64, dtype=torch.bfloat16, seed=S)
    out = sparda.decode_selected(y["q"].to(DEV), y["k_cache"].to(DEV), y["v_cache"].to(DEV), S, 64)
    nb = (S + 63) // 64
    sel = np.broadcast_to(np.arange(nb), (B, Hkv, nb))
    want = O.attention_decode(np32(y["q"]), np32(y["k_cache"]), np32(y["v_cache"]), S, sel,
                              np.full((B, Hkv), nb), 64)
    assert_close_out(np32(out), want, torch.bfloat16)


@pytest.mark.parametrize("first,last", [(64, 128), (256, 768), (0, 256), (0, 1000)])
def test_decode_dense_keys_at_minus_infinity(first, last):
    # a score of -inf weighs nothing, whether a block, a split or the sequence's head holds only such
    print(f"[case] decode dense -inf keys {first}..{last}", flush=True)
    S = 1500
    y = synth.decode_inputs(2, S, 12, 4, 64, dtype=torch.bfloat16, seed=S)
    q, k, v = y["q"].clone(), y["k_cache"].clone(), y["v_cache"]
    q[..., 0] = 1.0
    k[:, first:last, :, 0] = float("-inf")
    out = sparda.decode_selected(q.to(DEV), k.to(DEV), v.to(DEV), S, 64)
    keep = [s for s in range(S) if not first <= s < last]
    kk, vv = np32(k)[:, keep], np32(v)[:, keep]
    nb = (len(keep) + 63) // 64
    want = O.attention_decode(np32(q), kk, vv, len(keep), np.broadcast_to(np.arange(nb), (2, 4, nb)),
                              np.full((2, 4), nb), 64)
    assert_close_out(np32(out), want, torch.bfloat16)
