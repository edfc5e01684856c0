"""Build libblpg.so (HIP kernels + C ABI + C++ drop-in shim) in-tree for gfx950.

Usage: python -m simplexprojects_amd.build   (or simplexprojects_amd.build.build()).
Objects go to simplexprojects_amd/_build/, the library to simplexprojects_amd/libblpg.so.
"""
from __future__ import annotations

import concurrent.futures as cf
import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
ROOT = PKG.parent
CSRC = PKG / "csrc"
OBJ = PKG / "_build"
LIB = PKG / "libblpg.so"

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = os.environ.get("BLPG_ARCH", "gfx950")

# -ffp-contract=off: every FMA in the kernels is explicit, so tableau arithmetic matches
#   the CPU oracle operation for operation.
# packed-fp32-ops disabled: no v_pk_* FP32 instructions are generated.
HIPFLAGS = [
    "-mllvm", "-simplifycfg-sink-common=false",
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-fno-gpu-flush-denormals-to-zero", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", f"-I{ROOT / 'include'}",
]
CXXFLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", f"-I{ROOT / 'include'}"]

HIP_SOURCES = ["kernel_wave.hip", "kernel_stream.hip", "kernel_tile.hip", "kernel_tile64.hip",
               "kernel_verify.hip", "kernel_util.hip",
               "kernel_mlp.hip", "abi.cpp", "simplex_shim.cpp", "warmstart.cpp", "serve.cpp",
               "noalloc.cpp"]
SHIM_TEST = PKG / "test_shim"  # C++ drop-in test program (tests/cpp/test_shim.cpp)
CXX_SOURCES = ["gen.cpp"]


def _run(cmd: list[str]) -> None:
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"build step failed ({r.returncode}): {' '.join(cmd)}\n{r.stdout}")
    out = "\n".join(l for l in r.stdout.splitlines() if "packed-fp32-ops" not in l)
    if out.strip():
        print(out, file=sys.stderr)


def _listing(asm: Path):
    """(kernel, inside inline assembly?, line) of a device listing's instructions and of the
    comments in inline assembly."""
    kernel, own = "", False
    for line in asm.read_text().splitlines():
        if line.startswith("_Z") and ":" in line:
            kernel = line.split(":")[0]
        elif "#ASMSTART" in line:
            own = True
        elif "#ASMEND" in line:
            own = False
        elif line.startswith("\t") and (own or line[1:2] not in ".;"):
            yield kernel, own, line.strip()


def _registers(code: str, kind: str) -> set[int]:
    """Numbers of the registers v.. or a.. that an instruction (or its operands) names."""
    out = set()
    for m in re.finditer(rf"(?<![\w.]){kind}(?:(\d+)|\[(\d+):(\d+)\])", code):
        lo, hi = (m[1], m[1]) if m[1] else (m[2], m[3])
        out.update(range(int(lo), int(hi) + 1))
    return out


def _check_accumulators(asm: Path) -> None:
    """Kernels that keep tableau entries in accumulation registers name them in inline
    assembly only; the compiler must not place values of its own there in such a kernel."""
    uses: dict[str, dict[bool, str]] = {}
    for kernel, own, line in _listing(asm):
        if re.search(r"[ ,]a(\d|\[)", line.split(";")[0]):
            uses.setdefault(kernel, {})[own] = line
    for k, u in uses.items():
        if len(u) == 2:
            raise RuntimeError(f"{asm.name}: in {k} the compiler uses accumulation registers "
                               f"({u[False]}): give the kernel more vector registers")


def _check_operand_waits(asm: Path, states: int = 2) -> int:
    """Matrix instructions and lane swaps read a vector register at the earliest `states` wait
    states after a vector instruction wrote it.  The compiler keeps that distance between
    instructions it knows, not where one is inline assembly, so it is read from the listing
    (straight down: a branch only adds to it).  Returns the number of matrix instructions."""
    count = 0
    recent: list[tuple[int, set[int], str]] = []  # (wait states since, registers written, line)
    for kernel, _, line in _listing(asm):
        op, _, operands = line.split(";")[0].strip().partition(" ")
        if not op or op.startswith("."):
            continue
        matrix, swap = op.startswith("v_mfma"), op.startswith("v_permlane")
        count += matrix
        reads = _registers(operands.partition(",")[2] if matrix else operands, "v") if matrix or swap else set()
        for age, regs, writer in recent:
            if regs & reads:
                raise RuntimeError(f"{asm.name}: in {kernel} '{line}' reads a register {age} wait "
                                   f"states after '{writer}'")
        wait = int(operands, 0) + 1 if op == "s_nop" else 1
        recent = [(age + wait, regs, writer) for age, regs, writer in recent if age + wait < states]
        if op.startswith("v_") and not matrix:
            written = operands if swap else operands.partition(",")[0]
            recent.append((0, _registers(written, "v"), line))
    return count


def _check_wave(asm: Path) -> None:
    _check_accumulators(asm)
    if _check_operand_waits(asm) == 0:
        raise RuntimeError(f"{asm.name}: no matrix instruction")


def _check_blocks(asm: Path) -> int:
    """Kernels that keep their block of the tableau in the registers from a number on (a
    comment in their inline assembly names it) name them in inline assembly only: the compiler
    must stay below it everywhere else.  Returns the number of such kernels; every kernel of
    the listing has to be one."""
    first: dict[str, dict[str, int]] = {}
    used: dict[str, list[str]] = {}
    for kernel, own, line in _listing(asm):
        m = re.match(r"; block from v(\w+)(?: a(\w+))?", line) if own else None
        if m:  # (decimal or hexadecimal)
            first[kernel] = {kind: int(x, 0) for kind, x in zip("va", m.groups()) if x}
        elif not own:
            used.setdefault(kernel, []).append(line)
    for kernel, lines in used.items():
        if kernel not in first:
            raise RuntimeError(f"{asm.name}: {kernel} does not say where its block begins")
        for line in lines:
            code = line.split(";")[0]
            for kind, lim in first[kernel].items():
                if any(r >= lim for r in _registers(code, kind)):
                    raise RuntimeError(f"{asm.name}: in {kernel} the compiler uses registers of the "
                                       f"block, which begins at {kind}{lim} ({line})")
    return len(first)


# kernels whose registers inline assembly names, and what their listing has to keep
CHECKS = {"kernel_wave.hip": _check_wave, "kernel_tile.hip": _check_blocks,
          "kernel_tile64.hip": _check_blocks}


def _compile(src: Path) -> Path:
    obj = OBJ / (src.name + ".o")
    if src.name in CHECKS:
        _run([HIPCC, *HIPFLAGS, "--save-temps=obj", "-x", "hip", "-c", str(src), "-o", str(obj)])
        asm = list(OBJ.glob(f"{src.stem}-hip-*{ARCH}.s"))
        if len(asm) != 1:
            raise RuntimeError(f"{src.name}: no device assembly to check")
        CHECKS[src.name](asm[0])
        return obj
    if src.suffix == ".hip" or src.name in ("abi.cpp", "simplex_shim.cpp", "warmstart.cpp",
                                            "serve.cpp", "noalloc.cpp"):
        cmd = [HIPCC, *HIPFLAGS, "-x", "hip", "-c", str(src), "-o", str(obj)]
    else:
        cmd = ["g++", *CXXFLAGS, "-c", str(src), "-o", str(obj)]
    _run(cmd)
    return obj


def build(verbose: bool = False) -> Path:
    OBJ.mkdir(exist_ok=True)
    sources = [CSRC / s for s in HIP_SOURCES + CXX_SOURCES if (CSRC / s).exists()]
    jobs = min(len(sources), max(1, min(8, os.cpu_count() or 1)))
    with cf.ThreadPoolExecutor(jobs) as ex:
        objs = list(ex.map(_compile, sources))
    tmp = LIB.with_suffix(".so.tmp")
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", str(tmp),
          *map(str, objs), "-lpthread"])
    shutil.move(str(tmp), str(LIB))
    # the C++ drop-in test program links the library like a reference caller would
    _run(["g++", "-O1", "-std=c++17", f"-I{ROOT / 'include'}", str(ROOT / "tests/cpp/test_shim.cpp"),
          str(LIB), "-Wl,-rpath,$ORIGIN", "-o", str(SHIM_TEST)])
    if verbose:
        print(f"built {LIB}")
    return LIB


if __name__ == "__main__":
    build(verbose=True)
