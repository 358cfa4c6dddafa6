"""Compile-time checks of the gfx950 code (CPU only: hipcc cross-compiles without a GPU).

Every kernel of libpthdec.so must run without scratch memory: a spill to scratch in the decode
or prefill kernels costs a memory round trip per spilled value inside the tile loop. The check
compiles each kernel source to gfx950 assembly with the flags of the product build and reads
each kernel's `.private_segment_fixed_size` from the code-object metadata.
"""
import os
import re
import shutil
import subprocess
import sys

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
PKG_DIR = os.path.join(ROOT, "mi50-vllm-lab_amd")


def _hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    return None


@pytest.fixture(scope="module")
def gfx950_asm(tmp_path_factory):
    hipcc = _hipcc()
    if hipcc is None:
        pytest.skip("hipcc not available")
    sys.path.insert(0, PKG_DIR)
    try:
        import build as pd_build
    finally:
        sys.path.remove(PKG_DIR)
    flags = [f for f in pd_build.HIP_FLAGS if f not in ("-shared", "-fPIC")]
    tmp = tmp_path_factory.mktemp("asm")
    text = []
    for src in pd_build.KERNEL_SOURCES:
        out = str(tmp / (os.path.basename(src) + ".s"))
        cmd = [hipcc, *flags, "--cuda-device-only", "-S", "-I", os.path.join(ROOT, "include"), src, "-o", out]
        res = subprocess.run(cmd, capture_output=True, text=True)
        assert res.returncode == 0, (src, res.stderr[-4000:])
        with open(out) as f:
            text.append(f.read())
    return text


def _kernel_metadata(asms):
    """{kernel name: metadata text} from the amdhsa.kernels lists of the code objects."""
    out = {}
    for asm in asms:
        meta = asm[asm.index("amdhsa.kernels:"):]
        entries = re.split(r"\n  - ", meta)
        for e in entries[1:]:
            m = re.search(r"\.name:\s+(\S+)", e)
            if m:
                out[m.group(1)] = e
    return out


def test_every_kernel_is_built(gfx950_asm):
    names = _kernel_metadata(gfx950_asm)
    for k in ("pd_partial_kernel", "pd_combine_kernel", "pd_prefill_kernel", "pd_cache_write_kernel"):
        assert any(k in n for n in names), (k, sorted(names))
    # decode: one to three 16-row blocks, fast and general block-size paths
    assert sum("pd_partial_kernel" in n for n in names) == 6


def test_no_kernel_uses_scratch(gfx950_asm):
    meta = _kernel_metadata(gfx950_asm)
    scratch = {}
    for name, text in meta.items():
        m = re.search(r"\.private_segment_fixed_size:\s+(\d+)", text)
        assert m, name
        scratch[name] = int(m.group(1))
    assert all(v == 0 for v in scratch.values()), {k: v for k, v in scratch.items() if v}


def test_no_packed_fp32_instructions(gfx950_asm):
    # the build disables the packed-FP32 VALU forms; none may appear in the code
    for asm in gfx950_asm:
        assert not re.search(r"\bv_pk_(add|mul|fma)_f32\b", asm)


def _registers(operand):
    """{("v" or "a", number)} of a vector register operand, empty for any other."""
    m = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand.split(" ")[0])
    if not m:
        return set()
    first, last = (m.group(2), m.group(2)) if m.group(2) else m.group(3, 4)
    return {(m.group(1), i) for i in range(int(first), int(last) + 1)}


def early_matrix_reads(asm, states_needed):
    """(vector instruction, matrix instruction) pairs where the second reads what the first wrote fewer than
    `states_needed` (1 or 2) wait states before it."""
    found, recent = [], []  # recent: wait states and registers written, of the last instructions
    for line in asm.splitlines():
        text = line.split(";")[0].strip()
        if not re.match(r"[a-z]\w+(\s|$)", text) or text.endswith(":"):
            continue
        name, rest = (text.split(None, 1) + [""])[:2]
        operands = [x.strip() for x in re.split(r",(?![^\[]*\])", rest)]
        written = set()
        if name.startswith("v_mfma"):
            read, waited = set().union(*(_registers(x) for x in operands[1:4])), 0
            for states, regs, who in reversed(recent):
                if waited >= states_needed:
                    break
                if regs & read:
                    found.append((who, text))
                    break
                waited += states
        elif name.startswith("v_"):
            written = _registers(operands[0])
            if name.startswith(("v_permlane", "v_swap")):
                written |= _registers(operands[1])
        recent = recent[-2:] + [(int(operands[0]) + 1 if name == "s_nop" else 1, written, text)]
    return found


def test_matrix_operands_have_settled(gfx950_asm):
    # inline asm is outside the compiler's own hazard checks. The 256-row prefill writes operands and products both
    # in asm, so it keeps the two wait states between them itself; elsewhere the products are the compiler's
    close = ["v_cvt_f16_i16_sdwa v5, sext(v1) dst_sel:WORD_1", "s_nop 0", "v_mfma_f32_16x16x32_f16 a[0:3], v[2:5], v[8:11], a[0:3]"]
    close = "\n".join("\t" + x for x in close)
    assert len(early_matrix_reads(close, 2)) == 1 and not early_matrix_reads(close, 1)
    assert not early_matrix_reads(close.replace("s_nop 0", "s_nop 1"), 2)
    kernels = {}
    for asm in gfx950_asm:
        wide = "pd_prefill_wide_kernel" in asm
        kernels[wide] = kernels.get(wide, 0) + asm.count("v_mfma")
        assert early_matrix_reads(asm, 2 if wide else 1) == []
    assert kernels[True] > 0 and kernels[False] > 0


def test_halves_of_a_register_are_not_written_back_to_back(gfx950_asm):
    # a conversion that preserves the other half reads the register: one wait state after the one that wrote it
    for asm in gfx950_asm:
        last = ""
        for line in asm.splitlines():
            text = line.split(";")[0].strip()
            if not re.match(r"[a-z]\w+(\s|$)", text):
                continue
            if "UNUSED_PRESERVE" in text and "_sdwa" in last:
                assert text.split()[1] != last.split()[1], (last, text)
            last = text


def test_save_temps_takes_a_relative_directory(tmp_path, monkeypatch):
    # a stand-in compiler that writes its output where it runs and links only what is there
    cc = tmp_path / "hipcc"
    cc.write_text('#!/bin/sh\nfor a in "$@"; do case "$a" in *.o) [ "$last" = -o ] || [ -f "$a" ] || exit 3;; esac; last=$a; done\n'
                  'while [ "$1" != -o ]; do shift; done\necho built > "$2"\n')
    cc.chmod(0o755)
    monkeypatch.setenv("HIPCC", str(cc))
    monkeypatch.syspath_prepend(PKG_DIR)
    monkeypatch.chdir(tmp_path)
    import build as pd_build
    monkeypatch.setattr(pd_build, "LIB_DIR", str(tmp_path / "lib"))
    monkeypatch.setattr(pd_build, "LIB_PATH", str(tmp_path / "lib" / "libpthdec.so"))
    for d in ("temps", str(tmp_path / "absolute"), None):
        assert open(pd_build.build(d)).read() == "built\n"
        if d:
            assert len([f for f in os.listdir(tmp_path / d) if f.endswith(".o")]) == len(pd_build.SOURCES)
