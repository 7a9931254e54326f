"""Build libdsv2lite_hip.so for gfx950 with hipcc (in-tree, no JIT cache).

    python flash-deepseek-v2-lite_amd/csrc/build.py [-j N]

Each .hip file compiles to an object in parallel, then one shared library is
linked into ``flash-deepseek-v2-lite_amd/triton_kernels/``.  The library links
``libamdhip64.so.7``; loading it after ``import torch`` binds it to the HIP
runtime torch already loaded (same soname), so streams and graphs are shared.
"""

from __future__ import annotations

import argparse
import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import sys

CSRC = os.path.dirname(os.path.abspath(__file__))
PKG = os.path.dirname(CSRC)
ROOT = os.path.dirname(PKG)
INCLUDE = os.path.join(ROOT, "include")
OUT = os.path.join(PKG, "triton_kernels", "libdsv2lite_hip.so")
OBJDIR = os.path.join(PKG, "_build")
SOURCES = ["elementwise.hip", "gemv.hip", "gemm.hip", "mla.hip", "mla_small.hip", "moe.hip", "attention_expanded.hip", "mla_prefill.hip"]
ARCH = os.environ.get("DSV2_OFFLOAD_ARCH", "gfx950")

CXXFLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I", INCLUDE, "-I", CSRC,
    # packed-FP32 VALU ops off (v_pk_{add,mul,fma}_f32 are not emitted)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def hipcc() -> str:
    for c in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if c and os.path.exists(c):
            return c
    raise RuntimeError("hipcc not found (ROCm is required to build the HIP library)")


def _compile(src: str) -> str:
    obj = os.path.join(OBJDIR, src.replace(".hip", ".o"))
    asm = ASM_MFMA.get(src)
    cmd = [hipcc(), *CXXFLAGS, *(["--save-temps=obj"] if asm else []), "-c", os.path.join(CSRC, src), "-o", obj]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed for {src}:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    if asm:
        with open(os.path.join(OBJDIR, src.replace(".hip", f"-hip-amdgcn-amd-amdhsa-{ARCH}.s"))) as f:
            bad = mfma_hazards(f.read(), asm)
        if bad:
            os.remove(obj)
            raise RuntimeError(f"{src}: MFMA hazards the compiler does not see in inline asm:\n" + "\n".join(bad[:20]))
    return obj


# Kernels whose MFMAs are inline asm: the compiler's hazard recognizer takes an asm statement for
# one ordinary instruction, so the wait states around it are checked in the assembly it made.
ASM_MFMA = {"gemm.hip": "gemm_big_kernel"}
# wait states (an s_nop N counts N + 1, any other instruction 1): from an MFMA to an access of an
# accumulator by anything else -- the 16 passes of the longest bf16 form and the write behind them --
# and from a VALU write to an MFMA that reads the register
MFMA_TO_ACC, VALU_TO_MFMA = 19, 2


def _registers(operand: str) -> set[str]:
    """VGPRs and AGPRs an operand names: v3, v[4:7], a12, a[0:3]."""
    m = re.fullmatch(r"([va])(?:(\d+)|\[(\d+):(\d+)\])", operand)
    if not m:
        return set()
    lo, hi = (int(m[2]), int(m[2])) if m[2] else (int(m[3]), int(m[4]))
    return {f"{m[1]}{i}" for i in range(lo, hi + 1)}


def mfma_hazards(asm: str, kernel: str) -> list[str]:
    """Places in the functions whose symbol contains `kernel` that leave fewer wait states than
    MFMA_TO_ACC or VALU_TO_MFMA, along the code as laid out and over every branch."""
    funcs, cur = [], None
    for line in asm.split("\n"):
        head = re.match(r"(\w+):", line)
        if head and kernel in head[1] and not line.startswith("."):
            cur = (head[1], [], {})
            funcs.append(cur)
        elif cur is not None and line.startswith(".Lfunc_end"):
            cur = None
        elif cur is not None:
            label = re.match(r"(\.LBB\w+):", line)
            text = line.split(";")[0].strip()
            if label:
                cur[2][label[1]] = len(cur[1])
            elif text and not text.startswith("."):
                op, _, rest = text.partition(" ")
                cur[1].append((op, [x.strip() for x in rest.split(",")], text))
    bad: list[str] = []

    def scan(name: str, code: list) -> None:
        since_mfma, written = 1 << 20, {}  # wait states since an MFMA / since each register's VALU write
        for op, args, text in code:
            regs = [_registers(a) for a in args]
            if op.startswith("v_mfma"):
                for r in set().union(*regs[1:]):
                    if written.get(r, 1 << 20) < VALU_TO_MFMA:
                        bad.append(f"{name}: {r} written {written[r]} wait states before {text}")
                since_mfma = -1
            elif any(r[0] == "a" for rs in regs for r in rs) and since_mfma < MFMA_TO_ACC:
                bad.append(f"{name}: {since_mfma} wait states after an MFMA: {text}")
            states = int(args[0], 0) + 1 if op == "s_nop" else 1
            since_mfma += states
            written = {r: n + states for r, n in written.items() if n + states < VALU_TO_MFMA}
            if op.startswith("v_") and not op.startswith("v_mfma") and regs:
                written.update((r, 0) for r in regs[0])

    for name, code, labels in funcs:
        scan(name, code)
        for i, (op, args, _) in enumerate(code):
            if op.startswith("s_cbranch") or op == "s_branch":
                to = labels[args[0]]
                scan(f"{name} over {args[0]}", code[max(0, i - 2 * MFMA_TO_ACC):i + 1] + code[to:to + 2 * MFMA_TO_ACC])
    if not funcs:
        bad.append(f"no function named *{kernel}* in the assembly")
    elif not any(op.startswith("v_mfma") for _, code, _ in funcs for op, _, _ in code):
        bad.append(f"no MFMA in *{kernel}*")
    return list(dict.fromkeys(bad))


def _check_no_missing_stubs(lib: str) -> None:
    """A kernel whose host launch stub the compiler left undefined links into a library that
    only fails when it is loaded; refuse it at build time."""
    nm = shutil.which("nm")
    if not nm:
        return
    r = subprocess.run([nm, "-D", "--undefined-only", lib], capture_output=True, text=True)
    missing = [ln.split()[-1] for ln in r.stdout.splitlines() if "__device_stub__" in ln]
    if missing:
        os.remove(lib)
        raise RuntimeError(f"undefined kernel launch stubs in the linked library: {missing}")


def build(jobs: int | None = None, verbose: bool = False) -> str:
    os.makedirs(OBJDIR, exist_ok=True)
    jobs = jobs or min(len(SOURCES), os.cpu_count() or 4, 8)
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(_compile, SOURCES))
    tmp = OUT + ".tmp"
    # -Bsymbolic: the library's launches bind to its own kernel handles, never to a same-named
    # kernel of a library loaded before it with RTLD_GLOBAL (which would run that kernel on
    # this library's argument layout)
    cmd = [hipcc(), "-shared", "-fPIC", "-Wl,-Bsymbolic", f"--offload-arch={ARCH}", *objs, "-o", tmp]
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{r.stdout}\n{r.stderr}")
    _check_no_missing_stubs(tmp)
    os.replace(tmp, OUT)
    if verbose:
        print(f"built {OUT}", file=sys.stderr)
    return OUT


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("-j", type=int, default=None)
    a = ap.parse_args()
    build(a.j, verbose=True)
