"""The router's matrix-core scores against the oracle's fma chain, bit for bit:
row sets (alone and in pairs) and block chunks at their edges, every forecast
width, and forecasts with denormal, cancelling, infinite and NaN elements and of
mixed magnitude (where a chain differs from any other order of the sum)."""

import numpy as np
import pytest
import torch

import sparda
from oracle import sparda_oracle as O
from helpers import np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("Tq,NB,Df,k,causal,kind", [
    (1, 1, 64, 1, True, "normal"), (63, 2, 16, 2, True, "normal"), (65, 15, 32, 8, False, "normal"),
    (129, 17, 64, 8, True, "normal"), (200, 33, 128, 16, False, "normal"), (1000, 49, 64, 32, True, "normal"),
    (70, 3, 64, 4, False, "normal"), (70, 4, 64, 4, True, "normal"), (70, 5, 64, 8, False, "normal"),
    (70, 8, 64, 8, False, "normal"), (70, 9, 64, 8, False, "normal"), (70, 16, 128, 16, True, "normal"), (4161, 17, 16, 8, True, "normal"),
    (130, 70, 64, 8, False, "cancelling"), (130, 70, 128, 8, True, "mixed"), (130, 70, 16, 8, False, "mixed"),
    (130, 97, 64, 8, False, "tiny"), (130, 64, 64, 8, False, "infinite"), (130, 40, 64, 4, False, "equal")])
def test_route_scores_and_lists(Tq, NB, Df, k, causal, kind):
    print(f"[case] route Tq={Tq} NB={NB} Df={Df} {kind}", flush=True)
    g = torch.Generator().manual_seed(Tq + NB)
    H, bs = 3, 16
    f = torch.randn(2, Tq, H, Df, generator=g)
    p = torch.randn(2, NB, H, Df, generator=g)
    if kind == "tiny":
        f, p = f * 1e-20, p * 1e-20      # scores around 1e-39: denormal
    if kind == "cancelling":             # pairs of terms that leave a few bits, and sums that leave none
        f[..., 1::2], p[..., 1::2] = f[..., ::2], -p[..., ::2] * (1 + 2.0 ** -14)
        p[:, ::3, :, Df // 2:], f[..., Df // 2:] = -p[:, ::3, :, :Df // 2], f[..., :Df // 2]
    if kind == "mixed":                  # terms of 2^-40 to 2^40
        f = f * 2.0 ** torch.randint(-20, 21, f.shape, generator=g)
        p = p * 2.0 ** torch.randint(-20, 21, p.shape, generator=g)
    if kind == "infinite":
        p[:, ::7, :, 5] = float("inf")   # scores +inf or -inf
    if kind == "equal":
        p[:] = p[:, :1]                  # ties: the lower block first
    topk, scores, sel, n = sparda.route(f.to(DEV), p.to(DEV), bs, k, causal=causal, want_scores=True, want_sel=True)
    sc_o, tk_o, sel_o, n_o = O.route(np32(f), np32(p), bs, k, causal)
    assert np.array_equal(scores.cpu().numpy().view(np.int32), np.asarray(sc_o, np.float32).view(np.int32))
    assert np.array_equal(topk.cpu().numpy(), tk_o)
    assert np.array_equal(sel.cpu().numpy(), sel_o) and np.array_equal(n.cpu().numpy(), n_o)


def test_route_nan_scores_take_the_same_places():
    # a positive NaN ranks above every score, wherever the chain meets it
    print("[case] route NaN", flush=True)
    g = torch.Generator().manual_seed(3)
    f = torch.randn(1, 100, 2, 64, generator=g)
    p = torch.randn(1, 30, 2, 64, generator=g)
    p[:, 4, :, 9] = float("nan")
    p[:, 21, :, 63] = float("nan")
    topk = sparda.route(f.to(DEV), p.to(DEV), 64, 4, causal=False)[0].cpu().numpy()
    assert (topk[..., 0] == 4).all() and (topk[..., 1] == 21).all()
