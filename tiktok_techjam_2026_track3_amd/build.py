"""Build recipe for libmi355attn.so (gfx950 HIP kernels + C-ABI).

Compiles every ``csrc/*.hip`` to an object with hipcc (in parallel) and links the shared
library in-tree, next to this file, so it travels with the source tree. Run as
``python -m tiktok_techjam_2026_track3_amd.build``.
"""
from __future__ import annotations

import concurrent.futures as _cf
import os
import re
import shutil
import subprocess
import sys
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
CSRC = PKG_DIR / "csrc"
BUILD_DIR = PKG_DIR / "_build"
LIB_NAME = "libmi355attn.so"
LIB_PATH = PKG_DIR / LIB_NAME
ARCH = "gfx950"

# -ffp-contract=off: the int8 dequantisation must round multiply and add separately (it is
# compared bit for bit); kernels that want an FMA call __builtin_fmaf explicitly.
# -packed-fp32-ops disabled: packed fp32 VALU forms are not used anywhere in this library.
HIPCC_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the gfx950 kernels cannot be built")


def sources() -> list[Path]:
    return sorted(CSRC.glob("*.hip"))


# Kernels that issue LDS-DMA loads (buffer/global_load ... lds from inline assembly) and order
# them with hand-placed s_waitcnt / barriers. They must not use scratch memory: spill stores and
# reloads are vector-memory operations the hand-placed counts do not account for, and a spilling
# build of the attention loader produced nondeterministic rows. The build refuses such a kernel.
NO_SCRATCH_KERNELS = re.compile(r"attn_fwd_mfma|attn_fwd_tiled|attn_fwd_f32|gemm_kernel")
_REMARK = re.compile(r"remark:\s+(Function Name|ScratchSize \[bytes/lane\]|VGPRs Spill|SGPRs Spill):\s+(\S+)")


def resource_usage(stderr: str) -> dict:
    """kernel (mangled name) -> {"scratch": bytes per lane, "vgpr_spill": n, "sgpr_spill": n} from
    the compiler's -Rpass-analysis=kernel-resource-usage remarks."""
    out, cur = {}, None
    for m in _REMARK.finditer(stderr):
        key, val = m.group(1), m.group(2)
        if key == "Function Name":
            cur = out.setdefault(val, {})
        elif cur is not None:
            cur[{"ScratchSize [bytes/lane]": "scratch", "VGPRs Spill": "vgpr_spill",
                 "SGPRs Spill": "sgpr_spill"}[key]] = int(val)
    return out


def check_no_scratch(src_name: str, usage: dict) -> None:
    bad = [f"{name}: scratch {u.get('scratch')} B/lane, {u.get('vgpr_spill')} VGPR spills"
           for name, u in usage.items()
           if NO_SCRATCH_KERNELS.search(name) and (u.get("scratch", 0) or u.get("vgpr_spill", 0))]
    if bad:
        raise RuntimeError(f"{src_name}: LDS-DMA kernels must not use scratch memory:\n  "
                           + "\n  ".join(bad))


# The projection GEMM issues its MFMAs from inline assembly, where the compiler inserts no wait
# states. What it happens to emit around them has to keep these distances (in wait states: an
# instruction is one, s_nop n is n + 1), which the build checks in the device assembly:
ASM_MFMA_SOURCES = re.compile(r"gemm_(f16|bf16|f32|i8)$")
ASM_MFMA_KERNELS = re.compile(r"gemm_kernel")
VALU_TO_MFMA = 2  # a VGPR written by the vector ALU, then read by an MFMA
MFMA_TO_OTHER = 18  # an MFMA's result, then any other instruction on it (16 passes; these take 8)
_VREG = re.compile(r"\bv(?:(\d+)\b|\[(\d+):(\d+)\])")


def _vregs(text: str) -> set:
    out = set()
    for m in _VREG.finditer(text):
        lo, hi = (m[1], m[1]) if m[1] else (m[2], m[3])
        out.update(range(int(lo), int(hi) + 1))
    return out


def _hazards(seq: list) -> list:
    """Pairs of instructions of ``seq`` (in issue order) that are too close to each other."""
    bad, at, wrote, result = [], 0, {}, {}  # wrote / result: VGPR -> (wait state after it, text)
    for text in seq:
        op, _, args = text.partition(" ")
        if op == "s_nop":
            at += int(args, 0) + 1
            continue
        dst, _, src = args.partition(",")
        if op.startswith("v_mfma"):
            for r in _vregs(src):
                if r in wrote and at - wrote[r][0] < VALU_TO_MFMA:
                    bad.append((wrote[r][1], text))
            ab = ",".join(src.split(",")[:-1])  # A and B; C may be a result (the accumulator)
            for r in _vregs(ab):
                if r in result and at - result[r][0] < MFMA_TO_OTHER:
                    bad.append((result[r][1], text))
            for r in _vregs(dst):
                result[r] = (at + 1, text)
        else:
            for r in _vregs(args):
                if r in result and at - result[r][0] < MFMA_TO_OTHER:
                    bad.append((result[r][1], text))
            if op.startswith("v_"):
                for r in _vregs(dst):
                    wrote[r] = (at + 1, text)
        at += 1
    return bad


def mfma_hazards(asm: str) -> list:
    """(kernel, first instruction, second instruction) of every pair closer than the distances above
    in a unit's device assembly: along the text, and over every branch to its target."""
    out, kernel, code, labels = [], "", [], {}

    def flush():
        if not ASM_MFMA_KERNELS.search(kernel):
            return  # (builtin MFMAs: the compiler's own wait states)
        bad, start, reach = [], 0, 2 * MFMA_TO_OTHER
        for i, text in enumerate(code + ["s_endpgm"]):
            op, _, target = text.partition(" ")
            if op == "s_branch" or op.startswith("s_cbranch"):
                to = labels.get(target.strip())
                if to is not None:
                    bad += _hazards(code[max(start, i - reach):i + 1] + code[to:to + reach])
            if op in ("s_branch", "s_endpgm", "s_setpc_b64"):  # nothing falls through
                bad += _hazards(code[start:i])
                start = i + 1
        out.extend((kernel, a, b) for a, b in dict.fromkeys(bad))

    for line in asm.splitlines():
        text = line.split(";")[0].strip()
        if not text:
            continue
        label = re.match(r"([\w.$]+):", text)
        if label:
            if not label[1].startswith("."):
                kernel, code, labels = label[1], [], {}
            labels[label[1]] = len(code)
            if label[1].startswith(".Lfunc_end"):
                flush()
                code, labels = [], {}
        elif not text.startswith("."):
            code.append(" ".join(text.split()))
    return out


def check_mfma_hazards(src_name: str, asm: str) -> None:
    bad = mfma_hazards(asm)
    if bad:
        raise RuntimeError(f"{src_name}: {len(bad)} instruction pairs around inline MFMAs lack wait "
                           "states, first:\n  " + "\n  ".join(f"{k}: {a}  ->  {b}" for k, a, b in bad[:5]))


def _compile(src: Path) -> Path:
    obj = BUILD_DIR / (src.stem + ".o")
    check = ASM_MFMA_SOURCES.match(src.stem)
    cmd = [hipcc(), *HIPCC_FLAGS, "-Rpass-analysis=kernel-resource-usage",
           *(["-save-temps=obj"] if check else []), "-c", str(src), "-o", str(obj)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src.name}:\n{res.stdout}\n{res.stderr}")
    check_no_scratch(src.name, resource_usage(res.stderr))
    if check:
        temps = [p for p in BUILD_DIR.glob(f"{src.stem}*") if p != obj]
        asm = [p for p in temps if p.suffix == ".s" and "amdgcn" in p.name]
        check_mfma_hazards(src.name, "\n".join(p.read_text() for p in asm))
        if not any("v_mfma" in p.read_text() for p in asm):
            raise RuntimeError(f"{src.name}: no device assembly to check")
        for p in temps:
            p.unlink()
    return obj


def build(verbose: bool = True) -> Path:
    """Compile all HIP sources and link ``libmi355attn.so``; always rebuilds."""
    BUILD_DIR.mkdir(exist_ok=True)
    srcs = sources()
    if not srcs:
        raise RuntimeError(f"no HIP sources under {CSRC}")
    with _cf.ThreadPoolExecutor(max_workers=min(8, len(srcs))) as ex:
        objs = list(ex.map(_compile, srcs))
    tmp = LIB_PATH.with_suffix(".so.tmp")
    # --no-undefined: a kernel whose host-side launch stub was not emitted fails here, not at load
    cmd = [hipcc(), f"--offload-arch={ARCH}", "-shared", "-fPIC", "-Wl,--no-undefined",
           *map(str, objs), "-o", str(tmp)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError(f"link failed:\n{res.stdout}\n{res.stderr}")
    os.replace(tmp, LIB_PATH)
    if verbose:
        print(f"built {LIB_PATH} from {len(srcs)} sources", file=sys.stderr)
    return LIB_PATH


if __name__ == "__main__":
    build()
