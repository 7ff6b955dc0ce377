"""Wait states behind the fp16 lo halves of tiled::split8, which inline asm writes: the compiler keeps
one before any vector instruction that reads such a result, an MFMA needs two.  In code built from the
header, and in the built library."""
import os
import re
import struct
import subprocess

import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "ming-tts_amd", "csrc")
LIB = os.path.join(CSRC, "libmingtts_hip.so")
ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
PROBE = """#include "tiled_kernel.hpp"
using namespace mt;
__global__ void split_then_mfma(const float *x, const tiled::u32x4t *b, float *o) {
    float v[8];
    for (int e = 0; e < 8; e++) v[e] = x[8 * threadIdx.x + e];
    tiled::u32x4t hi, lo;
    tiled::split8<DT_F16, true>(v, hi, lo);
    tiled::f32x16t c;
    for (int r = 0; r < 16; r++) c[r] = 0.0f;
    c = tiled::mfma32x<DT_F16>(lo, b[threadIdx.x], c);
    for (int r = 0; r < 16; r++) o[16 * threadIdx.x + r] = c[r];
}
"""


def _regs(op):
    m = re.fullmatch(r"-?\|?v\[(\d+):(\d+)\]\|?", op) or re.fullmatch(r"-?\|?v(\d+)\|?", op)
    return set() if not m else set(range(int(m[1]), int(m[m.lastindex]) + 1))


def short_waits(lines):
    """(writer, reader) pairs with too few wait states between a v_fma_mixhi_f16 and a vector
    instruction (1) or MFMA (2) that reads its result.  A branch target in between ends a search."""
    found = []
    ins = [l.split("//")[0].split(";")[0].strip() for l in lines]
    ins = [l for l in ins if l and not l.startswith(".")]
    for i, w in enumerate(ins):
        if not w.startswith("v_fma_mixhi_f16"):
            continue
        dst, states = _regs(w.split(None, 1)[1].split(",")[0].strip()), 0
        for r in ins[i + 1:i + 4]:
            if r.endswith(":") or states >= 2:
                break
            name, _, ops = r.partition(" ")
            ops = [o.strip() for o in ops.split(",")]
            need = 2 if name.startswith("v_mfma") else 1 if name.startswith("v_") else 0
            # the mixed fmas of a pair write halves of one register and read the other half as it is
            reads = set().union(*(_regs(o.split()[0]) for o in ops[1:] if o)) if need else set()
            if states < need and dst & reads:
                found.append((w, r))
            states += int(ops[0], 0) + 1 if name == "s_nop" else 1
    return found


def test_the_check_finds_a_short_wait():
    hi = "v_fma_mixhi_f16 v5, v1, 1.0, -v2 op_sel:[0,0,1] op_sel_hi:[0,0,1]"
    mfma = "v_mfma_f32_32x32x16_f16 v[8:23], v[4:7], v[24:27], 0"
    assert short_waits([hi, "s_nop 0", mfma]) and short_waits([hi, "v_mov_b32_e32 v9, v5"])
    assert not short_waits([hi, "s_nop 1", mfma]) and not short_waits([hi, "s_nop 0", "v_mov_b32_e32 v9, v5"])
    assert not short_waits([hi, "v_mov_b32_e32 v9, v6", "v_mov_b32_e32 v9, v6", mfma])


def test_split8_before_an_mfma(tmp_path):
    src, out = tmp_path / "probe.hip", tmp_path / "probe.s"
    src.write_text(PROBE)
    subprocess.run([f"{ROCM}/bin/hipcc", "--offload-arch=gfx950", "-O3", "-std=c++17", "-Xclang", "-target-feature", "-Xclang",
                    "-packed-fp32-ops", f"-I{CSRC}", f"-I{os.path.join(CSRC, '..', '..', 'include')}", "--cuda-device-only",
                    "-S", str(src), "-o", str(out)], check=True, capture_output=True)
    lines = out.read_text().splitlines()
    assert any("v_fma_mixhi_f16" in l for l in lines) and any("v_mfma" in l for l in lines)
    assert not short_waits(lines)


def test_built_library(tmp_path):
    """Every code object of the built library (the offload bundles of its object files)."""
    if not os.path.exists(LIB):
        pytest.skip("the library is not built")
    data, at, seen = open(LIB, "rb").read(), 0, 0
    magic = b"__CLANG_OFFLOAD_BUNDLE__"
    while (at := data.find(magic, at)) >= 0:
        n, p = struct.unpack_from("<Q", data, at + len(magic))[0], at + len(magic) + 8
        for _ in range(n):
            off, size, tl = struct.unpack_from("<QQQ", data, p)
            triple, p = data[p + 24:p + 24 + tl], p + 24 + tl
            code = data[at + off:at + off + size]
            if b"gfx950" not in triple or code[:4] != b"\x7fELF":
                continue
            f = tmp_path / "code.o"
            f.write_bytes(code)
            asm = subprocess.run([f"{ROCM}/llvm/bin/llvm-objdump", "-d", "--no-show-raw-insn", "--no-leading-addr", str(f)],
                                 check=True, capture_output=True, text=True).stdout.splitlines()
            seen += sum("v_fma_mixhi_f16" in l for l in asm)
            assert not short_waits(asm)
        at += len(magic)
    assert seen > 0
