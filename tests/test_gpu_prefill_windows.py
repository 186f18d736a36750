"""The block-sparse prefill over its query windows (16, 32, 64 and 128 tokens,
chosen by how many windows a call has): the routed launch against route +
prefill bit for bit, and the output against the float64 oracle, at the lengths
on either side of each change of window."""

import numpy as np
import pytest
import torch

import sparda
from sparda import synth
from oracle import sparda_oracle as O
from helpers import assert_close_out, np32

pytestmark = pytest.mark.gpu
DEV = "cuda"


@pytest.mark.parametrize("Hq,T,bs,k", [
    (12, 3, 64, 8), (12, 17, 32, 4), (4, 130, 64, 8),       # 16-token windows
    (12, 1280, 64, 8), (12, 1281, 64, 8),                   # 16 | 32
    (8, 2560, 32, 4), (16, 2561, 32, 4),                    # 32 | 64
    (12, 5120, 64, 8), (4, 5121, 64, 8), (16, 5121, 64, 8)  # 64 | 128 (four heads per group stay at 64)
])
def test_routed_prefill_on_either_side_of_a_window_change(Hq, T, bs, k):
    print(f"[case] windows Hq={Hq} T={T} bs={bs} k={k}", flush=True)
    x = synth.prefill_inputs(1, T, Hq, 4, 64, dtype=torch.bfloat16, seed=900 + T)
    d = {n: t.to(DEV) for n, t in x.items()}
    protos = sparda.compress(d["k"], bs)
    _, _, sel, n = sparda.route(d["forecast"], protos, bs, k, want_topk=False, want_sel=True)
    _, _, sel_o, n_o = O.route(np32(x["forecast"]), O.compress(np32(x["k"]), bs), bs, k, True)
    assert np.array_equal(sel.cpu().numpy(), sel_o)
    out = sparda.prefill(d["q"], d["k"], d["v"], sel, n, bs)
    got, sel2, n2 = sparda.prefill_routed(d["q"], d["k"], d["v"], d["forecast"], protos, bs, k, want_sel=True)
    assert torch.equal(sel2, sel) and torch.equal(n2, n) and torch.equal(got, out)
    r = np.random.default_rng(T)
    rows = sorted({(0, int(t)) for t in r.integers(0, T, 24)} | {(0, t) for t in (0, T // 2, T - 1)})
    want = O.attention_prefill(np32(x["q"]), np32(x["k"]), np32(x["v"]), sel_o, n_o, bs, True, rows=rows)
    mask = np.zeros(want.shape, bool)
    for b, t in rows:
        mask[b, t] = True
    assert_close_out(np32(got), want, torch.bfloat16, mask)
