"""Builds the two in-tree shared objects with hipcc, for gfx950 only.

  lib/libminfer_attn.so                      HIP kernels behind the C ABI of include/minfer_attn.h
  minfer/kernels/torch_ext/_C.so             PyTorch stable-ABI op registration calling that C ABI

The reference builds its extension through torch's CUDAExtension (reference: setup.py:65-84);
here hipcc is driven directly so that no source translation step is involved.
"""
import os
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB_DIR = os.path.join(HERE, "lib")
EXT_DIR = os.path.join(HERE, "minfer", "kernels", "torch_ext")
CORE_SO = os.path.join(LIB_DIR, "libminfer_attn.so")
EXT_SO = os.path.join(EXT_DIR, "_C.so")

HIP_FLAGS = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-fvisibility=hidden",
             "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-I" + os.path.join(ROOT, "include"), "-I" + CSRC]
KERNEL_SOURCES = ["attn_prefill.hip", "attn_decode.hip", "rope.hip", "rmsnorm.hip", "gemm.hip", "gemm_tile_f16.hip", "gemm_tile_bf16.hip", "quant.hip", "calib.hip", "attn_api.hip"]


def _run(cmd):
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if res.returncode != 0:
        sys.stderr.write(" ".join(cmd) + "\n" + res.stdout)
        raise RuntimeError("build step failed: " + cmd[0])
    return res.stdout


def asm_hazards(asm_text):
    """Distances the compiler cannot keep because one end is inside an asm statement, looked for in the device code:
    (1) a global->LDS copy (always emitted from asm here) whose scalar address pair was written by a vector instruction
        (readfirstlane / readlane) fewer than five instructions earlier;
    (2) a matrix instruction that reads a register (an operand's or its accumulator's) written inside an asm statement fewer than
        two issue slots earlier, or, when the matrix instruction is itself inside one, written by any vector instruction
        that close in front of it;
    (3) an instruction outside asm statements that touches an accumulation register fewer than 18 issue slots after a matrix
        instruction inside one wrote it (16x16x32: 11 are needed).
    Returns a list of (function, offending instruction, the write it follows too closely)."""
    import re
    found, func, window, in_asm = [], "?", [], False

    def regs(text, bank):
        out = set()
        for m in re.finditer(r"\b%s(?:\[(\d+):(\d+)\]|(\d+)\b)" % bank, text):
            out.update((bank, r) for r in (range(int(m.group(1)), int(m.group(2)) + 1) if m.group(1) else (int(m.group(3)),)))
        return out

    def acc_regs(text):
        return regs(text, "a")

    def vector_regs(text):
        return regs(text, "v") | regs(text, "a")

    def written(text):
        operands = text.split(None, 1)[1] if len(text.split()) > 1 else ""
        return vector_regs(operands if "swap" in text.split()[0] else operands.split(",", 1)[0])

    def issue_slots(text):   # s_nop N fills N + 1
        n = re.match(r"s_nop (\d+)", text)
        return int(n.group(1)) + 1 if n else 1

    for raw in asm_text.split("\n"):
        line = raw.strip()
        if line.startswith(";;#ASMSTART"):
            in_asm = True
            continue
        if line.startswith(";;#ASMEND"):
            in_asm = False
            continue
        if not line or line.startswith((";", "//")):
            continue
        if line.endswith(":") or (":" in line and line.split(":")[0].replace("_", "").replace(".", "").replace("$", "").isalnum() and " " not in line.split(":")[0]):
            label = line.split(":")[0]
            if not label.startswith(".L"):
                func, window = label, []
            continue   # a branch target keeps the window: whatever path leads here, these instructions may have just run
        if line.startswith("."):
            continue
        op = line.split()[0]
        if op == "global_load_lds_dwordx4":
            m = re.search(r"s\[(\d+):(\d+)\]", line)
            if m:
                pair = {int(m.group(1)), int(m.group(2))}
                states = 0   # issue slots between the write and this instruction
                for prev, _ in reversed(window):
                    if states >= 5:
                        break
                    w = re.match(r"v_read(?:first)?lane_b32 s(\d+)", prev)
                    if w and int(w.group(1)) in pair:
                        found.append((func, line, prev))
                    states += issue_slots(prev)
        elif op.startswith("v_mfma"):
            srcs, states = vector_regs(line.split(",", 1)[1] if "," in line else ""), 0
            for prev, prev_in_asm in reversed(window):
                if states >= 2:
                    break
                if prev.startswith("v_") and not prev.startswith("v_mfma") and (prev_in_asm or in_asm):
                    if srcs & written(prev):
                        found.append((func, line, prev))
                states += issue_slots(prev)
        if not in_asm and window:
            touched = acc_regs(line)
            states = 0
            for prev, prev_in_asm in reversed(window) if touched else ():
                if states >= 18:
                    break
                if prev_in_asm and prev.startswith("v_mfma") and touched.intersection(acc_regs(prev.split(",", 1)[0])):
                    found.append((func, line, prev))
                states += issue_slots(prev)
        window.append((line, in_asm))
        if len(window) > 20:
            window.pop(0)
        if op in ("s_branch", "s_endpgm"):
            window = []   # what stands next in the text does not run next
    return found


def scratch_users(asm_text):
    """Kernels whose registers did not suffice: (name, bytes of scratch memory per lane) of those that have any."""
    import re
    sizes = re.findall(r"^    \.name:\s*(\S+)\n    \.private_segment_fixed_size:\s*(\d+)$", asm_text, flags=re.M)
    return [(name, int(size)) for name, size in sizes if int(size)]


def build_core(verbose=False):
    os.makedirs(LIB_DIR, exist_ok=True)
    obj_dir = os.path.join(HERE, "build")
    os.makedirs(obj_dir, exist_ok=True)
    objs = [os.path.join(obj_dir, s.replace(".hip", ".o")) for s in KERNEL_SOURCES]
    asms = [os.path.join(obj_dir, s.replace(".hip", ".s")) for s in KERNEL_SOURCES]
    cmds = [["hipcc", *HIP_FLAGS, "-c", os.path.join(CSRC, s), "-o", o] for s, o in zip(KERNEL_SOURCES, objs)]
    # the same device code as text, for the scan below (the objects' code is the same compilation's)
    cmds += [["hipcc", *HIP_FLAGS, "--cuda-device-only", "-S", os.path.join(CSRC, s), "-o", a] for s, a in zip(KERNEL_SOURCES, asms)]
    with ThreadPoolExecutor(max_workers=os.cpu_count() or 8) as ex:
        outs = list(ex.map(_run, cmds))
    if verbose:
        print("".join(outs))
    for a in asms:
        with open(a) as f:
            text = f.read()
        bad = asm_hazards(text)
        if bad:
            raise RuntimeError("asm statement too close to an instruction that depends on it in %s:\n%s" % (
                os.path.basename(a), "\n".join("  %s: %s  <-  %s" % b for b in bad[:20])))
        if scratch_users(text):   # (every kernel here is meant to fit its registers: set-up alone is felt by the short calls)
            raise RuntimeError("scratch memory in %s:\n%s" % (os.path.basename(a), "\n".join("  %s: %d bytes" % u for u in scratch_users(text))))
    _run(["hipcc", "--offload-arch=gfx950", "-shared", "-fPIC", "-o", CORE_SO, *objs])
    return CORE_SO


def build_torch_ext():
    import torch
    tdir = os.path.dirname(torch.__file__)
    tinc = os.path.join(tdir, "include")
    tlib = os.path.join(tdir, "lib")
    pyinc = sysconfig.get_paths()["include"]
    cmd = ["hipcc", "-O2", "-std=c++17", "-fPIC", "-shared", "-x", "c++",
           "-DUSE_ROCM", "-D__HIP_PLATFORM_AMD__", "-DPy_LIMITED_API=0x030a0000",
           "-DTORCH_TARGET_VERSION=0x020a000000000000",
           "-I" + os.path.join(ROOT, "include"), "-I" + tinc, "-I" + pyinc,
           os.path.join(CSRC, "torch_ops.cpp"), "-o", EXT_SO,
           "-L" + LIB_DIR, "-lminfer_attn", "-Wl,-rpath,$ORIGIN/../../../lib",
           "-L" + tlib, "-ltorch", "-ltorch_cpu", "-lc10", "-Wl,-rpath," + tlib]
    _run(cmd)
    return EXT_SO


def build_all(verbose=False):
    return build_core(verbose), build_torch_ext()


if __name__ == "__main__":
    for so in build_all(verbose=True):
        print("built", os.path.relpath(so, ROOT))
