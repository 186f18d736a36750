"""The fp32 matrix-core prefill (D = 64): group sizes, ragged tiles and blocks,
dense and listed, causal and not, lists with repeats (also on the general kernel,
reached through a block size of 16) against the float64 oracle (max-abs 1e-4, the
fp32 bar); infinite or NaN values of V that a token does not attend."""

import numpy as np
import pytest
import torch

import sparda
from sparda import _lib, synth
from oracle import sparda_oracle as O
from helpers import assert_close_out, np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("R,T,bs,k,causal,dense", [
    (1, 33, 64, 8, True, False), (3, 65, 32, 4, True, False), (3, 333, 64, 2, True, False),
    (4, 200, 32, 4, False, False), (5, 190, 64, 8, True, False), (16, 130, 32, 4, True, False),
    (3, 127, 64, 8, True, True), (2, 97, 64, 8, False, True), (3, 1, 64, 8, True, True),
    # either side of the lengths the general kernel keeps
    (3, 40, 64, 8, True, False), (3, 41, 64, 8, True, True), (3, 41, 64, 8, True, False), (1, 16, 32, 4, True, False),
    (1, 17, 32, 4, False, False), (8, 10, 64, 8, True, False), (8, 11, 64, 8, False, False)])
def test_f32_prefill_against_the_oracle(R, T, bs, k, causal, dense):
    print(f"[case] f32 R={R} T={T} bs={bs} causal={causal} dense={dense}", flush=True)
    x = synth.prefill_inputs(2, T, 2 * R, 2, 64, dtype=torch.float32, seed=60 + T)
    d = {n: t.to(DEV) for n, t in x.items()}
    sel = n = sel_o = n_o = None
    if not dense:
        _, _, sel, n = sparda.route(d["forecast"], sparda.compress(d["k"], bs), bs, k, causal=causal, want_topk=False,
                                    want_sel=True)
        sel_o, n_o = sel.cpu().numpy(), n.cpu().numpy()
    out = sparda.prefill(d["q"], d["k"], d["v"], sel, n, bs, causal=causal)
    want = O.attention_prefill(np32(x["q"]), np32(x["k"]), np32(x["v"]), sel_o, n_o, bs, causal)
    assert_close_out(np32(out), want, torch.float32)


@pytest.mark.parametrize("bs,R,cap", [
    (64, 3, 3), (16, 3, 3),                       # matrix-core and general kernel
    (64, 1, 40), (64, 3, 112), (32, 16, 700),     # every entry of a wide list in use
    (16, 2, 150)])
def test_f32_prefill_repeated_and_out_of_range_entries(bs, R, cap):
    # the allowed keys are a set: a repeat counts once, an entry outside the blocks not at all
    print(f"[case] f32 repeats bs={bs} R={R} cap={cap}", flush=True)
    T, Hkv = 260, 2
    x = synth.prefill_inputs(1, T, R * Hkv, Hkv, 64, dtype=torch.float32, seed=4)
    r = np.random.default_rng(5)
    sel = r.integers(-1, (T + bs - 1) // bs + 1, (1, Hkv, T, cap)).astype(np.int32)
    sel[..., 0] = 0
    sel[..., 2] = np.where(r.random((1, Hkv, T)) < 0.5, sel[..., 1], sel[..., 2])
    n = r.integers(1, 4, (1, Hkv, T)).astype(np.int32) if cap == 3 else np.full((1, Hkv, T), cap, np.int32)
    q, k, v, s_d, n_d = (t.to(DEV) for t in (x["q"], x["k"], x["v"], torch.from_numpy(sel), torch.from_numpy(n)))
    got = sparda.prefill(q, k, v, s_d, n_d, bs)
    want, _ = O.attention_prefill_masked(np32(x["q"]), np32(x["k"]), np32(x["v"]), sel, n, bs)  # lists as sets
    assert_close_out(np32(got), want, torch.float32)


def test_f32_prefill_rows_in_descending_order():
    # a negative token stride of K and V at the C entry (the first row is the last in memory)
    print("[case] f32 negative stride", flush=True)
    T, Hq, Hkv = 130, 6, 2
    x = {n: t.to(DEV) for n, t in synth.prefill_inputs(1, T, Hq, Hkv, 64, dtype=torch.float32, seed=9).items()}
    want = sparda.prefill(x["q"], x["k"], x["v"], None, None, 64)
    q, k, v = x["q"], x["k"].flip(1).contiguous(), x["v"].flip(1).contiguous()
    st, out = Hkv * 64, torch.empty_like(want)
    end = 4 * st * (T - 1)
    _lib.call("sparda_prefill", q.data_ptr(), *q.stride()[:3], k.data_ptr() + end, v.data_ptr() + end, T * st, -st, 64,
              _lib.F32, None, None, 0, 1, T, Hq, Hkv, 64, 64, 1, 0.125, out.data_ptr(), *out.stride()[:2],
              torch.cuda.current_stream().cuda_stream)
    assert (out - want).abs().max().item() < 1e-5


@pytest.mark.parametrize("bad", [float("inf"), float("nan")])
def test_f32_prefill_values_of_unattended_keys_stay_out(bad):
    print(f"[case] f32 V = {bad}", flush=True)
    T, at = 150, 70
    x = synth.prefill_inputs(1, T, 6, 2, 64, dtype=torch.float32, seed=8)
    v = x["v"].clone()
    v[0, at, :, 3] = bad
    q, k = x["q"].to(DEV), x["k"].to(DEV)
    clean = sparda.prefill(q, k, x["v"].to(DEV), None, None, 64)
    got = sparda.prefill(q, k, v.to(DEV), None, None, 64)
    assert (got[:, :at] - clean[:, :at]).abs().max().item() < 1e-5  # tokens before the key: as without it
    g = got.view(1, T, 6, 64)
    assert not torch.isfinite(g[:, at:, :, 3]).any()
    keep = [i for i in range(64) if i != 3]
    assert (g[..., keep] - clean.view(1, T, 6, 64)[..., keep]).abs().max().item() < 1e-5
