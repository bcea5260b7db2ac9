"""CPU check of the gfx950 assembly: the wait states between an MFMA and the reads of its result.

The hardware does not hold back a vector or memory instruction that reads an MFMA's result too early,
so 8 wait states (4-pass MFMAs) or 12 (8-pass) have to lie between them on every path.  The compiler
counts them, but not on every path into a merge of loops or switches; the kernels settle their
accumulators there (mfma_settle).  This walks every path of every kernel.
"""
from __future__ import annotations

import re

import pytest

from tests.test_isa_hazards import _kernels, _parse, isa  # noqa: F401  (isa is the module's fixture)

# Passes + 4 wait states; other MFMA shapes are not used.
NEED = {"v_mfma_f32_16x16x32_f16": 8, "v_mfma_f32_32x32x16_f16": 12, "v_mfma_i32_16x16x64_i8": 8}
STORES = ("ds_write", "global_store", "buffer_store", "global_atomic", "v_cmp", "v_readlane", "v_readfirstlane")


def _regs(tok: str):
    m = re.match(r"[-|]*([va])(?:\[(\d+):(\d+)\]|(\d+)\b)", tok)
    if not m:
        return frozenset()
    lo, hi = (int(m[2]), int(m[3])) if m[2] else (int(m[4]), int(m[4]))
    return frozenset((m[1], i) for i in range(lo, hi + 1))


def early_reads(lines):
    """Reads of an MFMA result, other than by an MFMA, before its wait states have passed."""
    ins, labels = _parse(lines)
    bad = []
    for k, (_, op, args, _, text) in enumerate(ins):
        if not op.startswith("v_mfma"):
            continue
        need = NEED[op]
        work, seen = [(k + 1, 0, _regs(args[0]))], set()
        while work:
            j, waited, live = work.pop()
            if j >= len(ins) or waited >= need or not live or (j, waited, live) in seen:
                continue
            seen.add((j, waited, live))
            _, o, a, _, t = ins[j]
            if o.startswith(("v_", "ds_", "global_", "buffer_", "flat_")) and a:
                src = a if o.startswith(STORES) else a[1:]
                if not o.startswith("v_mfma") and live & frozenset().union(*map(_regs, src)):
                    bad.append(f"{text} -> {t} after {waited}")
                    continue
                if not o.startswith(STORES):
                    live -= _regs(a[0])
            waited += int(a[0], 0) + 1 if o == "s_nop" else 1
            if o.startswith(("s_branch", "s_cbranch")) and a[0] in labels:
                work.append((labels[a[0]], waited, live))
            if not o.startswith(("s_branch", "s_endpgm")):
                work.append((j + 1, waited, live))
    return bad


def test_no_early_read_of_an_mfma_result(isa):  # noqa: F811
    ks = {k: v for k, v in _kernels(isa).items() if any("v_mfma" in t for t in v)}
    assert len(ks) >= 60
    bad = {k: b[:3] for k, b in ((k, early_reads(v)) for k, v in ks.items()) if b}
    assert not bad, bad


@pytest.mark.parametrize("nops,early", [(6, True), (7, False)])
def test_checker_counts_the_short_path(nops, early):
    """The failing pattern: a merge that one path reaches right after the MFMA."""
    lines = [".LBB0_1:", "v_mfma_f32_16x16x32_f16 v[4:7], v[8:11], v[12:15], v[4:7]", "s_cbranch_scc1 .LBB0_3",
             ".LBB0_2:", "s_nop 15", ".LBB0_3:", f"s_nop {nops - 1}", "v_mov_b32_e32 v0, v5", "s_cbranch_scc0 .LBB0_1",
             "s_endpgm"]
    assert bool(early_reads(lines)) is early
