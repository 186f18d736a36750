"""Wait states around hand-written cross-lane instructions, checked on the
code the compiler actually emits (CPU only: hipcc cross-compiles gfx950).

A VALU instruction with a DPP source, and a v_permlane16/32_swap, needs two
wait states after any VALU write of a VGPR it reads. The compiler inserts these
for the instructions it generates itself, but it does not count the results of
inline assembly as VALU writes, so the asm blocks carry their own s_nop
padding. What the compiler places between them (spill reloads, copies, index
arithmetic) is outside their control; this test compiles every source that
uses such inline assembly and checks each DPP / permlane-swap instruction of
every kernel against the rule.

A VALU instruction that reads a matrix-core result needs up to 20 wait states
after the product. The compiler places them for its own instructions and, again,
not for inline assembly: no VALU instruction of an asm block may read a register
that a product wrote fewer wait states before, on any path to it.
"""

import functools

import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG = os.path.join(ROOT, "local-research-small-language-model_amd")
sys.path.insert(0, PKG)
from sparda import build as B  # noqa: E402

WAIT_STATES = 2
MFMA_WAIT_STATES = 20  # the longest: VALU read after a product of 16 passes


def _vgprs(tok: str):
    tok = tok.strip()
    m = re.fullmatch(r"v(\d+)", tok)
    if m:
        return {int(m.group(1))}
    m = re.fullmatch(r"v\[(\d+):(\d+)\]", tok)
    if m:
        return set(range(int(m.group(1)), int(m.group(2)) + 1))
    return set()


def _operands(ins: str):
    parts = ins.split(None, 1)
    if len(parts) < 2:
        return []
    return [o.strip().split()[0] for o in parts[1].split(",") if o.strip()]


def _valu_writes(ins: str):
    op = ins.split()[0]
    if not op.startswith("v_"):
        return set()                        # SALU, memory and LDS results are not VALU writes
    ops = _operands(ins)
    if not ops:
        return set()
    if "swap" in op:                        # v_swap_b32, v_permlane*_swap write both operands
        out = set()
        for o in ops[:2]:
            out |= _vgprs(o)
        return out
    return _vgprs(ops[0])


def dpp_hazards(asm_lines):
    """List of (writer, dpp) pairs closer than WAIT_STATES; a label reached
    before the wait states are accounted for counts as a hazard too (the
    predecessor on another path is unknown)."""
    ins = []
    for l in asm_lines:
        s = l.split(";")[0].strip()
        if not s or s.startswith("."):
            if s.endswith(":"):
                ins.append(s)               # local labels such as .LBB3_4:
            continue
        ins.append(s)
    bad = []
    for i, l in enumerate(ins):
        op0 = l.split()[0]
        if l.endswith(":") or ("_dpp" not in op0 and "permlane" not in op0):
            continue
        reads = set()
        for o in _operands(l)[:3]:          # vdst (read by fmac / swap), src0, src1
            reads |= _vgprs(o)
        ws = 0
        for p in reversed(ins[max(0, i - 8):i]):
            if ws >= WAIT_STATES:
                break
            if p.endswith(":"):
                bad.append(("label " + p, l))
                break
            op = p.split()[0]
            if op == "s_nop":
                ws += int(p.split()[1], 0) + 1
                continue
            if _valu_writes(p) & reads:
                bad.append((p, l))
                break
            ws += 1
    return bad


def mfma_hazards(asm_lines):
    """List of (product, instruction): an inline-assembly VALU instruction that
    reads a result of the product fewer than MFMA_WAIT_STATES before, on some path."""
    ins, in_asm, labels, asm = [], [], {}, False
    for l in asm_lines:
        if "#ASMSTART" in l or "#ASMEND" in l:
            asm = "#ASMSTART" in l
            continue
        s = l.split(";")[0].strip()
        if not s or (s.startswith(".") and not s.endswith(":")):
            continue
        if s.endswith(":"):
            labels[s[:-1]] = len(ins)
        ins.append(s)
        in_asm.append(asm)
    preds = [[] for _ in ins]
    for i, s in enumerate(ins):
        op = s.split()[0]
        if op.startswith(("s_branch", "s_cbranch")):
            preds[labels[s.split()[1]]].append(i)
        if i + 1 < len(ins) and op not in ("s_branch", "s_endpgm", "s_setpc_b64"):
            preds[i + 1].append(i)
    bad = []
    for i, s in enumerate(ins):
        op = s.split()[0]
        if not in_asm[i] or not op.startswith("v_"):
            continue
        ops = _operands(s)
        if "swap" not in op and "fmac" not in op:
            ops = ops[1:]
        reads = frozenset().union(*(_vgprs(o) for o in ops))
        seen, todo = {}, [(j, reads, 0) for j in preds[i]]
        while todo:
            j, regs, ws = todo.pop()
            if ws >= MFMA_WAIT_STATES or seen.get((j, regs), MFMA_WAIT_STATES) <= ws:
                continue
            seen[(j, regs)] = ws
            p = ins[j]
            w = _valu_writes(p) & regs
            if w and p.startswith("v_mfma"):
                bad.append((p, s))
                break
            if not p.endswith(":"):
                ws += int(p.split()[1], 0) + 1 if p.startswith("s_nop") else 1
            if regs - w:
                todo += [(k, regs - w, ws) for k in preds[j]]
    return bad


def kernels(asm_text: str):
    """{kernel symbol: instruction lines} for every kernel in a device .s file."""
    out, cur = {}, None
    for l in asm_text.splitlines():
        m = re.match(r"^(_Z\S+):", l)
        if m:
            cur = m.group(1)
            out[cur] = []
            continue
        if cur is not None:
            # a kernel may end in several s_endpgm (early exits): read to its end label
            if l.startswith(".Lfunc_end"):
                cur = None
                continue
            out[cur].append(l)
    return out


def test_checker_flags_a_planted_hazard():
    planted = [
        "v_mov_b32_e32 v5, 0",
        "v_fmac_f32_dpp v5, v1, v2 row_newbcast:0 row_mask:0xf bank_mask:0xf",
    ]
    assert len(dpp_hazards(planted)) == 1
    swap = ["v_max_f32_e32 v4, v4, v5", "v_permlane16_swap_b32_e32 v4, v6"]
    assert len(dpp_hazards(swap)) == 1
    assert dpp_hazards([swap[0], "s_nop 1", swap[1]]) == []
    padded = [planted[0], "s_nop 1", planted[1]]
    assert dpp_hazards(padded) == []
    one_short = [planted[0], "s_nop 0", planted[1]]
    assert len(dpp_hazards(one_short)) == 1
    spill = ["v_accvgpr_read_b32 v2, a7", "v_add_u32_e32 v9, v9, v8", planted[1]]
    assert len(dpp_hazards(spill)) == 1
    unrelated = ["v_mov_b32_e32 v7, 0", planted[1]]
    assert dpp_hazards(unrelated) == []
    after_label = [".LBB0_3:", planted[1]]
    assert len(dpp_hazards(after_label)) == 1


def test_checker_flags_a_planted_read_of_a_product():
    mfma = "v_mfma_f32_16x16x32_bf16 v[0:3], v[8:11], v[12:15], 0"
    asm = lambda *l: [";;#ASMSTART", *l, ";;#ASMEND"]
    read = asm("v_max3_f32 v5, v1, v6, v7")
    assert len(mfma_hazards([mfma, *read])) == 1
    assert len(mfma_hazards([mfma, "s_nop 15", *read])) == 1
    assert mfma_hazards([mfma, "s_nop 15", "s_nop 3", *read]) == []
    assert mfma_hazards([mfma, "v_max_f32_e32 v1, 0, v2", *read]) == []          # the compiler's own read waits
    assert mfma_hazards([mfma, "v_max3_f32 v5, v1, v6, v7"]) == []               # not inline assembly
    # the product on the taken path only
    jump = ["s_cbranch_execz .LBB0_2", "s_nop 15", "s_nop 15", ".LBB0_2:", *read]
    assert len(mfma_hazards([mfma, *jump])) == 1
    assert mfma_hazards([mfma, "s_branch .LBB0_3", *jump, "s_endpgm", ".LBB0_3:", "s_endpgm"]) == []
    loop = [".LBB0_1:", *read, "s_nop 4", mfma, "s_cbranch_scc1 .LBB0_1"]
    assert len(mfma_hazards(loop)) == 1


def _dpp_sources():
    """Sources whose kernels use DPP or permlane-swap inline assembly (also
    through the shared headers)."""
    hdr = {h: open(os.path.join(B.CSRC, h)).read() for h in os.listdir(B.CSRC) if h.endswith(".h")}
    asm_hdr = [h for h, t in hdr.items() if re.search(r"asm\s*\(.*(_dpp|permlane)", t)]
    out = []
    for src in B.sources():
        text = open(src).read()
        if re.search(r"asm\s*\(.*(_dpp|permlane)", text) or any(f'"{h}"' in text for h in asm_hdr):
            out.append(src)
    return out


@functools.lru_cache(maxsize=None)
def _device_asm(src):
    r = subprocess.run([B.HIPCC, *B.FLAGS, "--cuda-device-only", "-S", os.path.join(B.CSRC, src), "-o", "-"],
                       capture_output=True, text=True)
    assert r.returncode == 0, r.stderr[-2000:]
    return kernels(r.stdout)


needs_hipcc = pytest.mark.skipif(shutil.which(B.HIPCC) is None and not os.path.exists(B.HIPCC),
                                 reason="hipcc not available")
SOURCES = [os.path.basename(s) for s in _dpp_sources()]


@needs_hipcc
@pytest.mark.parametrize("src", SOURCES)
def test_emitted_dpp_wait_states(src):
    n_dpp = 0
    problems = []
    for name, lines in _device_asm(src).items():
        n_dpp += sum(1 for l in lines if "_dpp" in l.split(";")[0] or "permlane" in l.split(";")[0])
        for w, d in dpp_hazards(lines):
            problems.append(f"{name[:60]}: {w} -> {d}")
    assert n_dpp > 0, "no DPP / permlane-swap instructions found; the check would be vacuous"
    assert not problems, "\n".join(problems[:20])


@needs_hipcc
@pytest.mark.parametrize("src", SOURCES)
def test_inline_assembly_waits_for_products(src):
    ks = _device_asm(src)
    if not any("v_mfma" in l for lines in ks.values() for l in lines):
        pytest.skip("no products in this source")
    assert any("#ASMSTART" in l for lines in ks.values() for l in lines), "no inline assembly found: vacuous"
    problems = [f"{name[:60]}: {w} -> {d}" for name, lines in ks.items() for w, d in mfma_hazards(lines)]
    assert not problems, "\n".join(problems[:20])
