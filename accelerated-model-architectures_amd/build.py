"""Offline build of libxma_rocm.so: hipcc cross-compiles the hand-written HIP
sources in csrc/ for gfx950 and links them into xma/rocm/libxma_rocm.so, which
the Python host loads with ctypes.  No torch headers, no JIT cache."""

from __future__ import annotations

import os
import re
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor


HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(os.path.dirname(HERE), "include")
OUT_DIR = os.path.join(HERE, "xma", "rocm")
LIB = os.path.join(OUT_DIR, "libxma_rocm.so")
SOURCES = ["grouped_gemm.hip", "grouped_gemm_f16.hip", "mid_rows.hip", "api.hip", "routing.hip", "elementwise.hip", "grouped_gemm_staged.hip", "fp32.hip", "router.hip", "gate.hip", "swiglu.hip", "bias.hip", "few_rows.hip", "layer.hip", "diagnostics.hip"]

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = [
    "-O3",
    "-std=c++17",
    "--offload-arch=gfx950",
    "-fPIC",
    "-fno-gpu-rdc",
    "-fvisibility=hidden",
    # keep the compiler from forming packed fp32 VALU ops
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    # per-kernel register, scratch and LDS figures on stderr (parsed below)
    "-Rpass-analysis=kernel-resource-usage",
    "-I", CSRC,
    "-I", INCLUDE,
]

# The grouped GEMM kernels read their fragments from LDS, and some of their row indices from memory, with inline assembly and
# wait for them by hand: between such a load and its wait the compiler takes the destination registers for ordinary values
# (or, if nothing uses them, for free ones), and whatever it does with them there meets data that arrives later.  The build
# therefore reads the generated ISA of those kernels and fails if any instruction that a path of the program leads to touches
# the destination of such a load before the wait, or if a loop of MFMAs without an inner loop accesses scratch memory (spills;
# those outside such loops are reported with the kernel's registers).  It also says so if the compiler is not the version the
# kernels were written and measured with.
CHECK_ISA = {"grouped_gemm.hip": re.compile(r"grouped_gemm"), "grouped_gemm_f16.hip": re.compile(r"grouped_gemm"), "mid_rows.hip": re.compile(r"mid_\w+_kernel")}
TESTED_HIPCC = "7.2"
USAGE_REPORT = os.path.join(HERE, "build", "kernel_resource_usage.txt")


def _registers(operands: str) -> set[str]:
    regs = set()
    for kind, lo, hi, kind1, n in re.findall(r"\b([va])\[(\d+):(\d+)\]|\b([va])(\d+)\b", operands):
        regs |= {f"{kind}{i}" for i in range(int(lo), int(hi) + 1)} if kind else {kind1 + n}
    return regs


class _Block:
    """basic block of a kernel: (line number, opcode, operands, inside inline assembly, text) per instruction, the indices of
    its successors, and the registers with a load in flight at its entry"""

    def __init__(self):
        self.code, self.succ, self.flight = [], [], {}


def _kernels(asm_path: str, which: re.Pattern):
    """(name, basic blocks in program order) of the kernels of a device ISA listing whose names match `which`"""
    name, blocks, labels, in_asm = None, [], {}, False
    with open(asm_path) as f:
        for n, line in enumerate(f, 1):
            label = re.match(r"^(_Z\w+|\.LBB\w+|\.Lfunc_end\w+):", line)
            if label and not label.group(1).startswith(".LBB"):
                if name:
                    for i, b in enumerate(blocks):
                        op, target = b.code[-1][1:3] if b.code else ("", "")
                        b.succ = [labels[target.strip()]] if op.startswith(("s_branch", "s_cbranch")) else []
                        if op not in ("s_branch", "s_endpgm", "s_setpc_b64") and i + 1 < len(blocks):
                            b.succ.append(i + 1)
                    yield name, blocks
                name = label.group(1) if which.search(label.group(1)) else None
                blocks, labels, in_asm = [_Block()], {}, False
                continue
            text = line.strip()
            if text.startswith(";;#ASM"):
                in_asm = text.startswith(";;#ASMSTART")
            if label and name:
                if blocks[-1].code:
                    blocks.append(_Block())
                labels[label.group(1)] = len(blocks) - 1
            elif name and text and text[0] not in ";.":
                op, _, operands = re.sub(r"\s+", " ", text.split(";")[0]).partition(" ")
                blocks[-1].code.append((n, op, operands, in_asm, text))
                if op.startswith(("s_branch", "s_cbranch", "s_endpgm", "s_setpc")):
                    blocks.append(_Block())


def _touched_in_flight(blocks: list[_Block]) -> list[str]:
    """instructions that touch the destination of an inline-assembly load from LDS or memory on some path before the wait
    behind it: s_waitcnt lgkmcnt(0) for LDS; for memory, where loads and stores retire in order, vmcnt(n) with at least n
    memory instructions behind the load on every path.  Fills in the blocks' `flight`: {(class, register): memory
    instructions behind the load, at least}"""

    def walk(block, bad):
        flight = dict(block.flight)
        for n, op, operands, in_asm, text in block.code:
            if op == "s_waitcnt":
                vm = re.search(r"vmcnt\((\d+)\)", operands)
                younger = int(vm.group(1)) if vm else 1 << 30
                flight = {f: c for f, c in flight.items() if ("lgkmcnt(0)" not in operands if f[0] == "ds" else c < younger)}
                continue
            regs = _registers(operands) if flight or in_asm else ()
            if any((c, r) in flight for r in regs for c in ("ds", "global")):
                bad.append((n, text))
            if op.startswith(("global_", "buffer_load", "buffer_store", "buffer_atomic", "scratch_", "flat_")):
                flight = {f: c if f[0] == "ds" else min(c + 1, 64) for f, c in flight.items()}
            if in_asm and (op.startswith("ds_read") or op.startswith("global_load") and "_lds" not in op):
                flight |= {(op.split("_")[0], r): 0 for r in _registers(operands.split(",")[0])}
        return flight

    todo = list(range(len(blocks)))
    while todo:
        block = blocks[todo.pop()]
        out = walk(block, [])
        for s in block.succ:
            merged = {f: min(c, blocks[s].flight.get(f, c)) for f, c in out.items()}
            if any(blocks[s].flight.get(f) != c for f, c in merged.items()):
                blocks[s].flight = blocks[s].flight | merged
                todo.append(s)
    bad: list[tuple[int, str]] = []
    for block in blocks:
        walk(block, bad)
    return [f"line {n}: {text}" for n, text in sorted(bad)]


def _scratch_in_mfma_loops(blocks: list[_Block]) -> list[str]:
    """scratch accesses in the loops that contain MFMAs and no inner loop"""
    pred: list[list[int]] = [[] for _ in blocks]
    for i, block in enumerate(blocks):
        for s in block.succ:
            pred[s].append(i)
    loops: dict[int, set[int]] = {}
    for tail, block in enumerate(blocks):
        for head in block.succ:
            if head <= tail:
                body, todo = loops.setdefault(head, {head}), [tail]
                while todo:
                    i = todo.pop()
                    if i not in body:
                        body.add(i)
                        todo += pred[i]
    bad = []
    for head, body in loops.items():
        code = [c for i in sorted(body) for c in blocks[i].code]
        if not any(h != head and h in body for h in loops) and any(c[1].startswith("v_mfma") for c in code):
            bad += [f"line {c[0]}: {c[4]}" for c in code if c[1].startswith("scratch_")]
    return bad


def _check_isa(asm_path: str, which: re.Pattern) -> None:
    for name, blocks in _kernels(asm_path, which):
        for what, bad in (("registers touched while a load into them is in flight", _touched_in_flight(blocks)),
                          ("scratch accesses inside an MFMA loop", _scratch_in_mfma_loops(blocks))):
            if bad:
                raise RuntimeError(f"{what}, {name}:\n  " + "\n  ".join(bad[:10]))


def _resource_usage_from_asm(asm_path: str) -> dict[str, dict[str, str]]:
    """{kernel: {field: value}} from the kernel metadata at the end of a device ISA listing (a compile with -save-temps
    prints no resource remarks, so the kernels that the check below exists for are read from their listing)"""
    keys = {".vgpr_count": "VGPRs", ".agpr_count": "AGPRs", ".private_segment_fixed_size": "ScratchSize [bytes/lane]",
            ".group_segment_fixed_size": "LDS Size [bytes/block]", ".vgpr_spill_count": "VGPR spills",
            ".sgpr_spill_count": "SGPR spills", ".sgpr_count": "SGPRs"}
    out: dict[str, dict[str, str]] = {}
    cur: dict[str, str] = {}
    with open(asm_path) as f:
        for line in f:
            m = re.match(r"^\s+(?:- )?(\.[a-z_]+):\s+(\S+)\s*$", line)
            if not m:
                continue
            key, val = m.group(1), m.group(2)
            if key == ".agpr_count":  # first field of a kernel's record
                cur = {}
            if key in keys:
                cur[keys[key]] = val
            elif key == ".name" and val.startswith("_Z"):
                out[val] = cur
    for v in out.values():  # the VGPR figure of the remarks counts both files, as the occupancy rule does
        v.setdefault("Occupancy [waves/SIMD]", str(max(1, 512 // max(int(v.get("VGPRs", "512")), 1))))
    return out


def _resource_usage(stderr: str) -> dict[str, dict[str, str]]:
    """{kernel: {field: value}} from the -Rpass-analysis=kernel-resource-usage remarks"""
    out: dict[str, dict[str, str]] = {}
    cur = None
    for line in stderr.splitlines():
        m = re.search(r"remark:\s+(Function Name|[A-Za-z ]+(?: \[[^\]]*\])?):\s*(\S+)", line)
        if not m:
            continue
        key, val = m.group(1).strip(), m.group(2)
        if key == "Function Name":
            cur = out.setdefault(val, {})
        elif cur is not None:
            cur[key] = val
    return out


def _check_compiler(verbose: bool) -> None:
    r = subprocess.run([HIPCC, "--version"], capture_output=True, text=True)
    m = re.search(r"HIP version:\s*(\S+)", r.stdout)
    version = m.group(1) if m else "unknown"
    if not version.startswith(TESTED_HIPCC):
        print(f"build.py: warning: hipcc {version}, the kernels were written and measured with {TESTED_HIPCC}.x; "
              f"re-run the GPU parity tests before trusting this build", file=sys.stderr)
    elif verbose:
        print(f"hipcc {version}", flush=True)


def _compile(src: str, verbose: bool, defines: tuple[str, ...] = (), tag: str = "") -> str:
    obj = os.path.join(HERE, "build", src.replace(".hip", tag + ".o"))
    # keeps the device ISA next to the object (named after the source, so only the untagged build of a file may do this)
    extra = ["-save-temps=obj"] if src in CHECK_ISA and not tag else []
    cmd = [HIPCC, *FLAGS, *extra, *defines, "-c", os.path.join(CSRC, src), "-o", obj]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    noise = "is not a recognized feature for this target"
    usage = _resource_usage(r.stderr)
    err = "\n".join(l for l in r.stderr.splitlines() if noise not in l and "kernel-resource-usage" not in l)
    err = re.sub(r"(?m)^\s*\d+ \|.*\n\s*\| \^\s*$\n?", "", err)  # source excerpts under the remarks
    if r.returncode != 0:
        raise RuntimeError(f"hipcc failed on {src}:\n{err}")
    if re.search(r"warning|error", err) and verbose:
        print(err, file=sys.stderr)
    if extra:
        asm = os.path.join(HERE, "build", src.replace(".hip", "-hip-amdgcn-amd-amdhsa-gfx950.s"))
        _check_isa(asm, CHECK_ISA[src])
        usage = _resource_usage_from_asm(asm)
    return obj, usage


def build(verbose: bool = False) -> str:
    os.makedirs(os.path.join(HERE, "build"), exist_ok=True)
    os.makedirs(OUT_DIR, exist_ok=True)
    _check_compiler(verbose)
    with ThreadPoolExecutor(max_workers=4) as pool:
        results = list(pool.map(lambda s: _compile(s, verbose), SOURCES))
    objs = [o for o, _ in results]
    with open(USAGE_REPORT, "w") as f:
        for _, usage in results:
            for k, v in usage.items():
                spills = f" spilled VGPRs {v['VGPR spills']}" if v.get("VGPR spills", "0") != "0" else ""
                f.write(f"{k}: VGPRs {v.get('VGPRs')} AGPRs {v.get('AGPRs')} scratch {v.get('ScratchSize [bytes/lane]')} "
                        f"LDS {v.get('LDS Size [bytes/block]')} occupancy {v.get('Occupancy [waves/SIMD]')}{spills}\n")
    cmd = [HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", LIB, *objs]
    if verbose:
        print(" ".join(cmd), flush=True)
    r = subprocess.run(cmd, capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    return LIB


TIMING_LIB = os.path.join(OUT_DIR, "libxma_rocm_timing.so")


def build_timing(verbose: bool = False, rebuild: bool = True) -> str:
    """A second library for diagnostics/tile_phases.py: grouped_gemm.hip compiled with -DXMA_PST_TIMING (the persistent
    GEMM kernel stamps the real-time counter and the shader clock counter at six points of every tile and behind every K
    step of one tile), linked with the objects of the normal build (rebuild=False: those of the last build()).
    Not part of build(): nothing in the product loads it."""
    if rebuild:
        build(verbose)
    obj, _ = _compile("grouped_gemm.hip", verbose, ("-DXMA_PST_TIMING",), "_timing")
    objs = [obj if s == "grouped_gemm.hip" else os.path.join(HERE, "build", s.replace(".hip", ".o")) for s in SOURCES]
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", TIMING_LIB, *objs], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"link failed:\n{r.stderr}")
    return TIMING_LIB


if __name__ == "__main__":
    if "--timing-only" in sys.argv[1:]:
        print(build_timing(verbose=True, rebuild=False))
    else:
        print(build_timing(verbose=True) if "--timing" in sys.argv[1:] else build(verbose=True))
