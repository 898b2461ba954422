"""Build the gfx950 HIP library ``liboxr_verify.so`` in-tree.

Every ``csrc/*.hip`` file is compiled to an object with hipcc for gfx950 and the
objects are linked into one shared library next to this file.  The library
exports only the ``extern "C"`` entry points declared in ``include/oxr_verify.h``.

Flags that matter for results:

- ``-ffp-contract=off``: no fused multiply-add where the reference rounds a
  product and a sum separately.
- ``-fhip-fp32-correctly-rounded-divide-sqrt``: fp32 ``/`` and ``sqrtf`` are
  correctly rounded (the RMSNorm ``rsqrt`` is ``1 / sqrt``).
- ``-Xclang -target-feature -Xclang -packed-fp32-ops``: no packed fp32 VALU
  instructions (``v_pk_*_f32``), which have given intermittently wrong results
  on this machine pool.

Every kernel must run without scratch memory: the build reads the compiler's
resource-usage remarks and fails if any kernel has a nonzero ``ScratchSize``.
Several kernels wait on hand-counted vector-memory counts (``s_waitcnt vmcnt``)
that hold only while no compiler-inserted scratch traffic shares the counter,
and a spill would also cost the register budget the designs are sized for.

Sources that load blocks into LDS with inline asm (``dma_block`` in common.h)
are also compiled to assembly, and the build fails where the generated code
breaks what the compiler cannot check for such a load (``dma_faults``).

Usage: ``python oxr-inference_amd/build.py`` (or ``__graft_entry__.build()``).
"""

from __future__ import annotations

import concurrent.futures
import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

PACKAGE_DIR = Path(__file__).resolve().parent
REPO_DIR = PACKAGE_DIR.parent
CSRC = PACKAGE_DIR / "csrc"
BUILD_DIR = REPO_DIR / "_build"
LIB_NAME = "liboxr_verify.so"
LIB_PATH = PACKAGE_DIR / LIB_NAME
ARCH = "gfx950"

HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall",
    "-Wno-unused-function",
    f"-I{REPO_DIR / 'include'}",
]


def hipcc() -> str:
    for candidate in (os.environ.get("HIPCC"), shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if candidate and Path(candidate).exists():
            return candidate
    raise RuntimeError("hipcc not found: the gfx950 library cannot be built")


_NAME = re.compile(r"remark: Function Name: (\S+)")
_SCRATCH = re.compile(r"remark:\s+ScratchSize \[bytes/lane\]: (\d+)")


def scratch_users(remarks: str) -> list[tuple[str, int]]:
    """(kernel, bytes per lane) for every kernel whose resource-usage remark reports scratch."""
    users, name = [], None
    for line in remarks.splitlines():
        if m := _NAME.search(line):
            name = m.group(1)
        elif (m := _SCRATCH.search(line)) and name is not None and int(m.group(1)) > 0:
            users.append((name, int(m.group(1))))
    return users


_SGPRS = re.compile(r"\bs(?:\[(\d+):(\d+)\]|(\d+)\b)")
# Vector instructions that write a scalar register: as their first operand, or as the carry after it.
_WRITES_FIRST = re.compile(r"v_(readfirstlane|readlane|cmpx?)_")
_WRITES_SECOND = re.compile(r"v_(\w+_co_|div_scale_|mad_[iu]64_)")
_BASE_STATES = 5  # wait states from a vector write of a scalar register to a load that reads it


def _sgprs(operand: str) -> set[int]:
    found = set()
    for lo, hi, one in _SGPRS.findall(operand):
        found |= set(range(int(lo), int(hi) + 1)) if lo else {int(one)}
    return found


def dma_faults(asm: str) -> list[str]:
    """What a ``dma_block`` load needs and the compiler does not look after, where the assembly of a
    source breaks it: m0 is used by these loads alone, each right behind its own write of m0, and no
    vector instruction writes the load's base address in the 5 wait states before it (along every way
    there: blocks that fall through to it and blocks that branch to it)."""
    lines = [text for raw in asm.splitlines() if (text := raw.split(";")[0].strip())
             and not (text.startswith(".") and not text.endswith(":"))]
    branches: dict[str, list[int]] = {}
    for i, text in enumerate(lines):
        if text.startswith(("s_branch", "s_cbranch")):
            branches.setdefault(text.split()[-1], []).append(i)
    faults, blessed = [], set()

    def writes(text: str, base: set[int]) -> bool:
        operands = text.split(None, 1)[1].split(",") if " " in text or "\t" in text else []
        return bool((_WRITES_FIRST.match(text) and operands and _sgprs(operands[0]) & base)
                    or (_WRITES_SECOND.match(text) and len(operands) > 1 and _sgprs(operands[1]) & base))

    def written_above(i: int, states: int, base: set[int]) -> bool:
        """Whether ``base`` is written by line ``i`` or above it, within ``states`` wait states."""
        while i >= 0 and states > 0:
            text = lines[i]
            if text.endswith(":"):
                if any(written_above(j, states, base) for j in branches.get(text[:-1], ())):
                    return True
                if i and lines[i - 1].startswith(("s_branch", "s_endpgm", "s_setpc")):
                    return False  # nothing falls through to the label
            elif writes(text, base):
                return True
            else:
                states -= int(text.split()[1], 0) + 1 if text.startswith("s_nop") else 1
            i -= 1
        return False

    for i, text in enumerate(lines):
        if text.startswith("global_load_lds_dwordx4"):
            if i < 2 or not lines[i - 1].startswith("s_nop") or not lines[i - 2].startswith("s_mov_b32 m0,"):
                faults.append(f"load into LDS without its own write of m0: {text}")
                continue
            blessed.add(i - 2)
            base = _sgprs(text.split(",", 1)[1])
            if not base:
                faults.append(f"load into LDS from a base in other than numbered registers: {text}")
            elif written_above(i - 1, _BASE_STATES, base):
                faults.append(f"vector write of the base address just before: {text}")
    faults += [f"m0 used elsewhere: {text}" for i, text in enumerate(lines)
               if re.search(r"\bm0\b", text) and i not in blessed]
    return faults


def _check_dma(source: Path) -> None:
    if "dma_block" not in source.read_text():
        return
    cmd = [hipcc(), *HIPCC_FLAGS, "-S", "--cuda-device-only", str(source), "-o", "-"]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc -S failed for {source.name}:\n{proc.stderr}")
    faults = dma_faults(proc.stdout)
    if faults:
        raise RuntimeError(f"{source.name}: unsafe loads into LDS:\n" + "\n".join(f"  {f}" for f in faults))


def _compile(source: Path) -> Path:
    obj = BUILD_DIR / (source.stem + ".o")
    cmd = [hipcc(), *HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage", "-c", str(source), "-o", str(obj)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"hipcc failed for {source.name}:\n{' '.join(cmd)}\n{proc.stdout}{proc.stderr}")
    users = scratch_users(proc.stderr)
    if users:
        obj.unlink(missing_ok=True)
        listing = "\n".join(f"  {name}: {size} bytes/lane" for name, size in users)
        raise RuntimeError(f"{source.name}: kernels use scratch memory (register spills), not allowed:\n{listing}")
    return obj


def build(verbose: bool = False) -> Path:
    """Compile every kernel source and link ``liboxr_verify.so``; return its path."""
    BUILD_DIR.mkdir(exist_ok=True)
    sources = sorted(CSRC.glob("*.hip"))
    if not sources:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    workers = min(len(sources), int(os.environ.get("MAX_JOBS", os.cpu_count() or 4)), 16)
    with concurrent.futures.ThreadPoolExecutor(max_workers=max(workers, 1)) as pool:
        checks = [pool.submit(_check_dma, source) for source in sources]
        objects = list(pool.map(_compile, sources))
        for check in checks:
            check.result()
    tmp = LIB_PATH.with_suffix(".so.tmp")
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", *map(str, objects), "-o", str(tmp)]
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        raise RuntimeError(f"link failed:\n{' '.join(cmd)}\n{proc.stdout}{proc.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(sources)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build(verbose=True)
