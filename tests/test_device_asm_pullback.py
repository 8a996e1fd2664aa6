"""The assembly of the four-wave pull-back kernels, every one that the library holds (no GPU: hipcc cross-compiles).  Their MFMAs are inline assembly with tied
accumulators, so the compiler inserts no wait states in front of a read of a result by another unit, or of an operand, the accumulator
among them, that the vector ALU has just written (at least two): between an MFMA and the first
read of a register it wrote there must be at least 13 (what the compiler leaves behind the same MFMA as a builtin; every instruction counts as one,
another MFMA as the 8 for which it holds the matrix core, `s_nop n` as n + 1).  Inside the loops no accumulator is
moved and no load is waited for but by the loop's own count: a reload or a move there is what the layout of registers avoids."""

import re
import subprocess

import pytest

from __graft_entry__ import PKG_DIR, _load_build_module

REG = re.compile(r"\b([av])(?:(\d+)\b|\[(\d+):(\d+)\])")
STORES = ("scratch_store", "global_store", "buffer_store", "ds_write", "flat_store")


def regs(text):
    for m in REG.finditer(text):
        for r in ([int(m.group(2))] if m.group(2) else range(int(m.group(3)), int(m.group(4)) + 1)):
            yield m.group(1) + str(r)


def closest_read(lines):
    written, n, worst = {}, 0, 99
    for t in lines:
        nop = re.match(r"s_nop (\d+)", t)
        n += int(nop.group(1)) + 1 if nop else 8 if "mfma" in t else 1
        ops = t.split(None, 1)[1] if " " in t else ""
        if "mfma" in t:
            for r in regs(ops.split(", ")[0]):
                written[r] = n
            continue
        for r in regs(ops if t.startswith(STORES) else ",".join(ops.split(",")[1:])):
            if r in written:
                worst = min(worst, n - written.pop(r))
        if not t.startswith(STORES):
            for r in regs(ops.split(",")[0]):
                written.pop(r, None)
    return worst


def operand_gap(lines):
    """Fewest wait states between a vector instruction's write and an assembly MFMA (tied or from 0) that reads it."""
    written, n, worst = {}, 0, 99
    for t in lines:
        nop = re.match(r"s_nop (\d+)", t)
        n += int(nop.group(1)) + 1 if nop else 1
        if not t.startswith("v_"):
            continue
        ops = t.split(None, 1)[1].split(", ")
        if "mfma" in t:
            for r in regs(", ".join(ops[1:4])):
                worst = min(worst, n - written.get(r, -99) - 1)
        else:
            for r in regs(ops[0]):
                written[r] = n
    return worst


def kernels(asm):
    for m in re.finditer(r"^(_ZN4w8a8\d+(?:bwd_dx_wide|gq_bwd_dx_wide)_kernel\S+):(.*?)^\.Lfunc_end", asm, re.M | re.S):
        yield m.group(1), m.group(2)


def instructions(text):
    return [t.split(";")[0].strip() for t in text.split("\n") if t.startswith("\t") and not t.strip().startswith((".", ";"))]


def test_the_count_itself():
    assert closest_read(["v_mfma_f32_32x32x16_bf16 a[0:15], v[0:3], v[4:7], a[0:15]", "s_nop 3", "v_accvgpr_read_b32 v9, a5"]) == 5
    assert operand_gap(["v_or_b32_e32 v7, v1, v2", "s_nop 1", "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], v[16:31]"]) == 2
    assert operand_gap(["v_accvgpr_write_b32 a31, 0", "v_mfma_f32_32x32x16_bf16 a[16:31], v[0:3], v[4:7], a[16:31]"]) == 0
    assert closest_read(["v_mfma_f32_32x32x16_bf16 v[0:15], v[20:23], v[24:27], v[0:15]", "v_mov_b32 v3, v40", "v_mov_b32 v41, v3"]) == 99


RANKS = (0, 1, 2, 4)  # 16-wide rank blocks
TEMPLATES = [f"template __global__ void w8a8::gq_bwd_dx_wide_kernel<{w4},{terms},{nkk}>(GqBwdDxArgs);\n"
             for w4 in ("true", "false") for terms in (2, 3) for nkk in RANKS]
TEMPLATES += [f"template __global__ void w8a8::bwd_dx_wide_kernel<{nkk}>(BwdDxArgs);\n" for nkk in RANKS]


def test_results_are_not_read_early(tmp_path):
    build = _load_build_module()
    try:
        hipcc = build.find_hipcc()
    except RuntimeError as e:  # pragma: no cover - the image ships hipcc
        pytest.skip(str(e))
    flags = [f for f in build.HIPCC_FLAGS if f not in ("-shared", "-fPIC") and not f.startswith("-Wl,")]
    procs = []
    for part in range(4):  # (at once: a minute for all)
        tu = tmp_path / f"pullback{part}.hip"
        tu.write_text('#include "w8a8_gq_bwd.h"\nusing namespace w8a8;\n' + "".join(TEMPLATES[part::4]))
        procs.append(subprocess.Popen([hipcc, *flags, "--cuda-device-only", "-S", "-I", str(PKG_DIR / "csrc"), str(tu), "-o",
                                       str(tu.with_suffix(".s"))], stderr=subprocess.PIPE, text=True))
    errors = [p.communicate()[1] for p in procs]
    assert [p.returncode for p in procs] == [0] * 4, errors
    found = [k for part in range(4) for k in kernels((tmp_path / f"pullback{part}.s").read_text())]
    assert len(found) == len(TEMPLATES)
    for name, text in found:
        assert closest_read(instructions(text)) >= 13, name
        assert operand_gap(instructions(text)) >= 2, name
        loops = 0
        for block in re.split(r"^\.LBB\S+:", text, flags=re.M):
            ins = instructions(block)
            ins = ins[:next((i for i, t in enumerate(ins) if t.startswith("s_cbranch")), len(ins))]
            if sum("mfma_f32" in t for t in ins) >= 32 and any("s_barrier" in t for t in ins):
                loops += 1
                assert not [t for t in ins if t.startswith(("v_accvgpr", "scratch"))], name
                assert {t for t in ins if "vmcnt" in t} <= {"s_waitcnt vmcnt(6)" if "gq" in name else "s_waitcnt vmcnt(7)"}, name
        assert loops >= 2, name  # tiles of eight row blocks, and of four
