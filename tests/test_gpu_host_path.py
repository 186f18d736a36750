"""The operators' native host path against their full Python path: the same
outputs bit for bit on the common forms (defaults and explicit options, strided
views, fp32 and bf16), and the same exceptions on what neither accepts."""

import pytest
import torch

import sparda
from sparda import _lib, ops, synth

pytestmark = pytest.mark.gpu
DEV = "cuda"


class Spy:
    """The native path, counting the calls it answered."""

    def __init__(self):
        self.host, self.taken = _lib.load_host(), []

    def __getattr__(self, name):
        def f(*a):
            r = getattr(self.host, name)(*a)
            if r is not None:
                self.taken.append(name)
            return r
        return f


def _both(monkeypatch, fn):
    monkeypatch.setattr(ops, "_host", _lib._NoHost())
    want = fn()
    spy = Spy()
    monkeypatch.setattr(ops, "_host", spy)
    return fn(), want, spy.taken


def _flat(x):
    if isinstance(x, (list, tuple)):
        return [t for y in x for t in _flat(y)]
    return [] if x is None else [x]


def _calls():
    x = {n: t.to(DEV) for n, t in synth.prefill_inputs(2, 300, 12, 4, 64, dtype=torch.bfloat16, seed=1).items()}
    q, k, v, f = x["q"], x["k"], x["v"], x["forecast"]
    kv = torch.stack((k, v), 3)  # interleaved: strided views of one buffer
    protos = sparda.compress(k, 64)
    topk = sparda.route(f, protos, 64, 8, causal=False)[0]
    y = {n: t.to(DEV) for n, t in synth.decode_inputs(3, 1500, 12, 4, 64, dtype=torch.bfloat16, seed=2).items()}
    dq, dk, dv, df = y["q"], y["k_cache"], y["v_cache"], y["forecast"]
    ws = sparda.DecodeWorkspace(DEV)
    ws.get(1 << 20)
    sums = torch.zeros(3, 24, 4, 64, device=DEV)
    sparda.block_sums(dk, 0, 1500, 64, sums)
    pos = torch.tensor([1499], device=DEV)
    g = torch.Generator().manual_seed(3)
    rnd = lambda *s: (0.05 * torch.randn(*s, generator=g)).to(torch.bfloat16).to(DEV)
    h, w, wo, wgu, wd = rnd(3, 1, 768), rnd(1536, 768), rnd(768, 768), rnd(4096, 768), rnd(768, 2048)
    cos, sin = torch.rand(1600, 32, device=DEV), torch.rand(1600, 32, device=DEV)
    kc, vc = dk.clone(), dv.clone()
    return {
        "compress": lambda: (sparda.compress(k, 64), sparda.compress(kv[:, :, :, 1], 48), sparda.compress(k.float(), 32)),
        "route": lambda: (sparda.route(f, protos, 64, 8), sparda.route(f, protos, 64, 32, False, scale=0.5)),
        "prefill": lambda: (sparda.prefill(q, k, v, None, None, 64),
                            sparda.prefill(q.float(), k.float(), v.float(), None, None, 64, causal=False, scale=0.2),
                            sparda.prefill(q, kv[:, :, :, 0], kv[:, :, :, 1], None, None, 32)),
        "prefill_routed": lambda: (sparda.prefill_routed(q, k, v, f, protos, 64, 8),
                                   sparda.prefill_routed(q, k, v, f.float(), protos, 64, 8, causal=False, scale=0.1,
                                                         route_scale=1)),
        "prefill_chunked": lambda: (sparda.prefill_chunked(q, k, v, topk, 64, 8),
                                    sparda.prefill_chunked(q, k, v, None, 64, 2, scale=0.3)),
        "decode": lambda: (sparda.decode(dq, dk, dv, 1500, df, 64, 8, workspace=ws),
                           sparda.decode(dq, dk, dv, 1337, df.float(), 32, 4, "absolute", workspace=ws),
                           sparda.decode(dq, dk, dv, 200, None, 64, 8, workspace=ws)),
        "decode_dense": lambda: (sparda.decode_selected(dq, dk, dv, 1500, 64),
                                 sparda.decode_selected(dq.float(), dk.float(), dv.float(), 77, 16, scale=0.2)),
        "decode_sums": lambda: (sparda.decode_sums(dq, dk, dv, 1500, df, sums, 64, 8, "absolute", pos_dev=pos,
                                                   update_current=True),
                                sparda.decode_sums(dq, dk, dv, 1400, df, sums, 64, 8)),
        "produce": lambda: (sparda.produce(h, w, 768, 256, 256, 1e-5, cos, sin, pos0=3, f_dtype=torch.float32),
                            sparda.produce(h, w, 768, 256, 256, 1e-5, cos, sin, pos_dev=pos),
                            sparda.produce(h, w, 768, 256, 256, 1e-5, cos, sin, pos_dev=pos, k_cache=kc, v_cache=vc),
                            kc[:, 1499], vc[:, 1499]),
        "ffn_decode": lambda: sparda.ffn_decode(h, wgu, wd, 1e-5),
        "rows_residual": lambda: (sparda.rows_residual(h, wo, h), sparda.rows_residual(q[:, :3].reshape(2, 3, 768), wo,
                                                                                     h.expand(3, 2, 768).transpose(0, 1))),
        "norm_gemv": lambda: sparda.norm_gemv(h, wgu, 1e-5),
        "teacher_mass": lambda: (sparda.teacher_block_mass(q, k), sparda.teacher_block_mass(q, k, causal=False, scale=0.3)),
    }


@pytest.mark.parametrize("name", ["compress", "route", "prefill", "prefill_routed", "prefill_chunked", "decode",
                                  "decode_dense", "decode_sums", "produce", "ffn_decode", "rows_residual", "norm_gemv",
                                  "teacher_mass"])
def test_native_path_equals_the_python_path(monkeypatch, name):
    print(f"[case] host path {name}", flush=True)
    with torch.no_grad():
        got, want, taken = _both(monkeypatch, _calls()[name])
    got, want = _flat(got), _flat(want)
    assert len(got) == len(want) and all(a.dtype == b.dtype and a.shape == b.shape and a.stride() == b.stride()
                                         and torch.equal(a, b) for a, b in zip(got, want))
    assert name in taken, "the native path answered none of the calls"


def test_refused_calls_raise_the_same(monkeypatch):
    print("[case] host path errors", flush=True)
    x = {n: t.to(DEV) for n, t in synth.prefill_inputs(1, 130, 12, 4, 64, dtype=torch.bfloat16, seed=1).items()}
    q, k, v, f = x["q"], x["k"], x["v"], x["forecast"]
    protos = sparda.compress(k, 64)
    ids = torch.zeros(1, 130, 4, 64, dtype=torch.int32, device=DEV)
    n = torch.ones(1, 4, 130, dtype=torch.int32, device=DEV)
    calls = [lambda: sparda.compress(k, 0), lambda: sparda.compress(ids, 64), lambda: sparda.compress(k.cpu(), 64),
             lambda: sparda.compress(k[0], 64), lambda: sparda.route(f, protos[:, :, :2], 64, 8),
             lambda: sparda.prefill(q, k.float(), v, None, None, 64), lambda: sparda.prefill(q[:, :, :11], k, v, None, None, 64),
             lambda: sparda.prefill_routed(q, k, v, f, protos, 32, 8), lambda: sparda.prefill_chunked(q, k, v, ids, 64, 8),
             lambda: sparda.decode_selected(q[:, 0], k, v, 131, 64), lambda: sparda.teacher_block_mass(q, k, 32),
             lambda: sparda.prefill(q, k, v, None, n, 64),
             lambda: sparda.decode_selected(q[:, 0], k, v, 130, 64, n_sel=n[:, :, 0]),
             lambda: sparda.ffn_decode(q, q, q, 1e-5), lambda: sparda.compress(k.requires_grad_(), 64)]
    for i, c in enumerate(calls):
        seen = []
        for host in (_lib._NoHost(), _lib.load_host()):
            monkeypatch.setattr(ops, "_host", host)
            with pytest.raises(Exception) as e:
                c()
            seen.append((e.type, str(e.value)))
        assert seen[0] == seen[1], (i, seen)
