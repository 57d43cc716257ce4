"""The attention kernels' inline-asm MFMA and DPP statements rely on the order of the compiled code instead of wait
states, which the compiler does not add for asm: in their assembly, along every branch too, no MFMA operand and no DPP
source is written by the VALU in the two instructions before, and no VGPR result of an MFMA is read or overwritten (by a
load either) before three more MFMAs were issued or 12 wait states passed, which is what the compiler puts behind the
same MFMA when it comes from a builtin."""
import os
import re
import subprocess

import pytest

from arcagi2_flashnext_dots3_amd import build

WAIT = 12
LOADS = ("ds_read", "global_load", "buffer_load", "scratch_load", "flat_load")
REG = re.compile(r"([av])(?:\[(\d+):(\d+)\]|(\d+))$")


def _regs(tok):
    m = REG.match(tok)
    if not m:
        return set()
    lo, hi = (m[4], m[4]) if m[4] else (m[2], m[3])
    return {(m[1], i) for i in range(int(lo), int(hi) + 1)}


def hazards(lines):
    """[(line, text)] of the violations in one kernel's assembly."""
    bad, hist, mfma, now = [], [], [], 0          # mfma: (destination, wait states issued before it)
    for n, l in enumerate(lines):
        l = l.split(";")[0].strip()
        if not l or l.startswith(".") or l.endswith(":"):
            continue
        op, _, rest = l.partition(" ")
        toks = [t.strip().split(" ")[0] for t in re.split(r",\s*(?![^\[]*\])", rest)]
        dst = _regs(toks[0])
        stores = op.startswith(("ds_write", "global_store", "scratch_store"))
        src = set().union(*map(_regs, toks if stores else toks[1:]))
        need = set().union(*map(_regs, toks[1:3])) if "mfma" in op else _regs(toks[1]) if "_dpp" in op else set()
        states = 0
        for o, d, imm in reversed(hist[-4:]):
            states += int(imm, 0) if o == "s_nop" else 0
            if o.startswith("v_") and "mfma" not in o and d & need and states < 2:
                bad.append((n, l))
            states += 1
        if "mfma" in op:
            mfma.append((dst, now))
        else:
            touched = {r for r in src | (dst if op.startswith(("v_", *LOADS)) else set()) if r[0] == "v"}
            if any(touched & d and now - at - 1 < WAIT for d, at in mfma[-3:]):
                bad.append((n, l))
        now += 1 + (int(toks[0], 0) if op == "s_nop" else 0)
        hist.append((op, set() if stores else dst, toks[0]))
    return bad


def branch_hazards(body, window=60):
    """The same over the code before and after every branch of the kernel's assembly."""
    labels = {l.split(":")[0]: i for i, l in enumerate(body) if re.match(r"\.LBB\w+:", l)}
    bad = []
    for i, l in enumerate(body):
        m = re.match(r"\s*s_c?branch\w*\s+(\.LBB\w+)", l)
        if m:
            j = labels[m[1]]
            bad += [(l.strip(), *b) for b in hazards(body[max(0, i - window):i + 1] + body[j:j + window])]
    return bad


def test_scanner_finds_planted_hazards():
    ok = ["v_add_f32_e32 v1, v2, v3", "s_nop 1", "v_mul_f32_dpp v4, v1, v5 quad_perm:[0,0,0,0]"]
    assert not hazards(ok)
    assert hazards([ok[0], ok[2]])
    m = "v_mfma_f32_32x32x16_bf16 v[16:31], v[0:3], v[4:7], 0"
    assert hazards(["v_mov_b32_e32 v5, v9", "s_nop 0", m])
    a = "v_mfma_f32_32x32x16_f16 a[0:15], v[40:43], v[44:47], a[0:15]"
    assert hazards([m, a, a, "ds_write_b128 v9, v[16:19] offset:64"])
    assert hazards([m, "s_nop 10", "v_add_f32_e32 v1, v16, v2"]) and not hazards([m, "s_nop 11", "v_add_f32_e32 v1, v16, v2"])
    assert hazards([m, "ds_read_b128 v[20:23], v9"]) and not hazards([m, "ds_read_b128 v[32:35], v9"])
    loop = [".LBB0_1:", "v_add_f32_e32 v1, v16, v2", "s_nop 15", m, "s_cbranch_scc1 .LBB0_1", "s_nop 15"]
    assert not hazards(loop) and branch_hazards(loop)
    skip = [m, "s_cbranch_scc1 .LBB0_2", "s_nop 15", ".LBB0_2:", "v_add_f32_e32 v1, v16, v2"]
    assert not hazards(skip) and branch_hazards(skip)
    assert not hazards([m, a, a, a, "ds_write_b128 v9, v[16:19] offset:64"])


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
@pytest.mark.parametrize("src,kernel,count", [("spmla_attn.hip", r"_ZN5spmla4attn10fwd_kernelI\S+:", 2),
                                              ("spmla_attn_hg.hip", r"_ZN5spmla2pk11attn_kernelI\S+:", 5)])
def test_compiled_order_of_asm_statements(tmp_path, src, kernel, count):
    out = tmp_path / "attn.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", os.path.join(build.CSRC, src), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text().split("\n")
    starts = [i for i, l in enumerate(text) if re.match(kernel, l)]
    assert len(starts) == count
    for s in starts:
        end = next(i for i in range(s, len(text)) if ".Lfunc_end" in text[i])
        body = text[s:end]
        assert sum("v_mfma_f32_32x32x16_bf16" in l for l in body) >= 36
        assert not hazards(body) and not branch_hazards(body)


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_wait_states_are_the_compilers(tmp_path):
    src = tmp_path / "m.hip"
    src.write_text("""#include <hip/hip_runtime.h>
typedef __bf16 bf16x8 __attribute__((ext_vector_type(8)));
typedef float f32x16 __attribute__((ext_vector_type(16)));
__global__ void k(const bf16x8* a, const bf16x8* b, f32x16* o) {
  o[threadIdx.x] = __builtin_amdgcn_mfma_f32_32x32x16_bf16(a[threadIdx.x], b[threadIdx.x], f32x16{}, 0, 0, 0) * 2.0f;
}
""")
    out = tmp_path / "m.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "--cuda-device-only", "-S", str(src), "-o", str(out)], check=True,
                   capture_output=True)
    m = re.search(r"v_mfma_f32_32x32x16_bf16 v.*\n\s*s_nop (\d+)", out.read_text())
    assert int(m[1]) + 1 <= WAIT


@pytest.mark.skipif(not os.path.exists(build.HIPCC), reason="no hipcc")
def test_chain_end_fills_the_wait(tmp_path):
    """chain_end alone is the whole wait, with nothing else in between."""
    src = tmp_path / "c.hip"
    src.write_text("""#include "spmla_attn_hg.hip"
__global__ void chain_probe(const bf16x8* a, const bf16x8* b, f32x16* o) {
  f32x16* dst = o + threadIdx.x;
  f32x16 c = spmla::pk::qk_first(a[threadIdx.x], b[threadIdx.x]);
  spmla::pk::chain_end<0>(c);
  *dst = c * 2.0f;
}
""")
    out = tmp_path / "c.s"
    subprocess.run([build.HIPCC, *build.FLAGS, "-I", build.CSRC, "--cuda-device-only", "-S", str(src), "-o", str(out)],
                   check=True, capture_output=True)
    text = out.read_text().split("\n")
    at = next(i for i, l in enumerate(text) if re.match(r"_Z11chain_probe\S+:", l))
    nops = re.findall(r"#ASMSTART\n\s*s_nop (\d+)\n", "\n".join(text[at:]))      # (the compiler's own nops not counted)
    assert int(nops[0]) + 1 >= WAIT
