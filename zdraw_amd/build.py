"""Builds the gfx950 shared libraries in-tree with hipcc / g++.

`python -m zdraw_amd.build` compiles
  zdraw_amd/lib/libzdraw_hip.so   the C-ABI library (HIP kernels + bridge)
  zdraw_amd/lib/libzdraw_host.so  the C++ host layer above the C ABI
hipcc cross-compiles for gfx950 without a GPU present.
"""
from __future__ import annotations

import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
HOST = os.path.join(HERE, "host")
LIBDIR = os.path.join(HERE, "lib")

HIP_LIB = os.path.join(LIBDIR, "libzdraw_hip.so")
HOST_LIB = os.path.join(LIBDIR, "libzdraw_host.so")

# Packed-FP32 VALU forms are disabled for every device translation unit.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]


def _run(cmd):
    proc = subprocess.run(cmd, capture_output=True, text=True)
    if proc.returncode != 0:
        sys.stderr.write(proc.stdout + proc.stderr)
        raise RuntimeError("build failed: " + " ".join(cmd))
    return proc


def build_hip(verbose: bool = False, out: str | None = None, extra_flags=()) -> str:
    """Compile the C-ABI library. `out` / `extra_flags` build an experimental
    copy elsewhere (kernel tuning defines) without touching the shipped one."""
    os.makedirs(LIBDIR, exist_ok=True)
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    target = out or HIP_LIB
    tag = "" if out is None else "." + os.path.basename(out)
    srcs = [os.path.join(CSRC, f) for f in ("attn_fwd.hip", "attn_wide.hip", "qk_prepass.hip", "gemm_half.hip", "bridge.hip")]
    from concurrent.futures import ThreadPoolExecutor
    objs = [os.path.join(LIBDIR, os.path.basename(src) + tag + ".o") for src in srcs]
    with ThreadPoolExecutor(max_workers=min(len(srcs), os.cpu_count() or 1)) as pool:  # one hipcc per source file
        list(pool.map(lambda so: _run([hipcc, *HIPCC_FLAGS, *extra_flags, "-c", so[0], "-o", so[1]]), zip(srcs, objs)))
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", target, *objs])
    if verbose:
        print("built", target)
    return target


_ASM_CACHE: dict = {}


def _device_asm(src: str, extra_flags=()) -> list[str]:
    import tempfile
    key = (src, tuple(extra_flags), os.path.getmtime(src))
    if key in _ASM_CACHE:
        return _ASM_CACHE[key]
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    with tempfile.TemporaryDirectory() as tmp:
        asm = os.path.join(tmp, "out.s")
        _run([hipcc, *HIPCC_FLAGS, *extra_flags, "-S", "--cuda-device-only", "-o", asm, src])
        with open(asm) as f:
            _ASM_CACHE[key] = f.read().split("\n")
    return _ASM_CACHE[key]


def m0_writes(src: str = os.path.join(CSRC, "gemm_half.hip"), kernels: str = "gemm_(ring|pipe)_kernel", extra_flags=()) -> list[str]:
    """Compiles `src` to gfx950 assembly and lists, for the kernels whose symbol matches
    `kernels`, every instruction that writes M0 other than the source's own
    `s_mov_b32 m0, <sgpr>` + `s_nop 0` pair (attn_device.hpp, lds_dma_base). The four-wave GEMMs
    keep M0 live across several loads without the compiler knowing; a write of the compiler's
    own in between would send those loads elsewhere in LDS."""
    import re
    lines = [l.split(";")[0].strip() for l in _device_asm(src, extra_flags)]
    lines = [l for l in lines if l]
    bad = []
    kernel = ""
    writes = re.compile(r"^s_\w+\s+m0\s*,")
    for i, text in enumerate(lines):
        if text.endswith(":") and not text.startswith("."):
            kernel = text[:-1]
            continue
        if not re.search(kernels, kernel) or not writes.match(text):
            continue
        own = re.match(r"^s_mov_b32\s+m0\s*,\s*s\d+$", text) and i + 1 < len(lines) and lines[i + 1] == "s_nop 0"
        if not own:
            bad.append(f"{kernel}: {text}")
    return bad


def tied_mfma_hazards(src: str = os.path.join(CSRC, "gemm_half.hip"), extra_flags=(),
                      mfma_prefix: str = "v_mfma_f32_16x16x32", kernel_substr: str = "") -> list[str]:
    """Compiles `src` to gfx950 assembly and lists every place (in the kernels whose symbol
    contains `kernel_substr`) where something other than an MFMA touches an accumulation
    register while a hand-written MFMA (`mfma_prefix`) may still be writing it. Those MFMAs are assembly statements, so the compiler adds none of
    the wait states it adds after the builtin; the source instead ends every run of them
    with `s_nop 15` before control leaves the block. A copy or spill of an accumulator that
    the register allocator places inside such a run would read a stale value: this check
    (run by the CPU tests) fails the build that contains one."""
    import re
    lines = _device_asm(src, extra_flags)
    bad = []
    agpr = re.compile(r"\ba(\[\d+:\d+\]|\d+)\b")
    kernel, hot = "", False
    for no, line in enumerate(lines, 1):
        text = line.split(";")[0].strip()
        if not text:
            continue
        if text.endswith(":") and not text.startswith("."):
            kernel, hot = text[:-1], False
            continue
        if kernel_substr not in kernel:
            continue
        op = text.split()[0]
        if op.startswith(mfma_prefix):
            hot = True
        elif op == "s_nop" and text.split()[1] == "15":
            hot = False
        elif hot and agpr.search(text):
            bad.append(f"{kernel}: line {no}: {text}")
    return bad


def vmem_sgpr_hazards(src: str, extra_flags=()) -> list[str]:
    """Compiles `src` to gfx950 assembly and lists every memory instruction that reads a scalar register
    which a vector instruction (v_readlane, v_readfirstlane, a compare into a register) wrote fewer than five wait states before. The
    hardware does not wait for such a write; the compiler keeps the distance for its own loads, not for the
    direct-to-LDS loads, which are assembly statements: with a stale descriptor or offset they would reach
    anywhere. Scalar registers restored from a spill ahead of such a load are the usual way to get there."""
    import re
    lines = [l.split(";")[0].strip() for l in _device_asm(src, extra_flags)]
    lines = [l for l in lines if l and (not l.startswith(".") or l.endswith(":"))]
    scalars = re.compile(r"\bs(?:(\d+)|\[(\d+):(\d+)\])")

    def registers(text):
        return {r for one, lo, hi in scalars.findall(text) for r in (range(int(one), int(one) + 1) if one else range(int(lo), int(hi) + 1))}

    bad, kernel = [], ""
    for i, text in enumerate(lines):
        if text.endswith(":") and not text.startswith("."):
            kernel = text[:-1]
        if not re.match(r"^v_\w+\s+s[\d\[]", text):
            continue
        written, states = registers(text.split(",")[0]), 0
        for later in lines[i + 1:i + 12]:
            # far enough, or written again by the scalar unit (compares and bit tests only read their first operand)
            if re.match(r"^s_(?!cmp|bitcmp)\w+\s+s[\d\[]", later):
                written -= registers(later.split(",")[0])
            if states >= 5 or not written:
                break
            if re.match(r"^(buffer|global|flat|scratch)_", later) and written & registers(later):
                bad.append(f"{kernel}: {text} | {states} wait states | {later}")
                break
            nop = re.match(r"^s_nop\s+(\d+)", later)
            states += int(nop.group(1)) + 1 if nop else 0 if later.endswith(":") else 1
    return bad


def kernarg_overreads(src: str, extra_flags=()) -> list[str]:
    """Compiles `src` to gfx950 assembly and lists every scalar load from a kernel's argument pointer that ends
    past the kernel's argument segment. The compiler sizes the segment by what the kernel declares and uses (the
    grid size and its like are there only in kernels that read them), not by loads that the source makes through the
    pointer itself (qk_prepass.hip, touch_args): nothing guarantees memory behind it."""
    import re
    lines = [l.split(";")[0].strip() for l in _device_asm(src, extra_flags)]
    sizes, first = {}, {}  # per kernel: bytes of the segment, first register of the pointer
    name = ""
    for text in lines:
        m = re.match(r"^\.amdhsa_(\w+)\s+(\S+)$", text)
        if not m:
            continue
        key, value = m.groups()
        if key == "kernel":
            name = value
            first[name] = 0
        elif key == "kernarg_size":
            sizes[name] = int(value)
        elif key in ("user_sgpr_dispatch_ptr", "user_sgpr_queue_ptr") and int(value):
            first[name] += 2  # these come ahead of it in the registers
    bad, kernel, pointers = [], "", set()
    for text in lines:
        m = re.match(r"^([\w$.]+):$", text)
        if m and not text.startswith("."):
            kernel = m.group(1)
            pointers = {first[kernel]} if kernel in first else set()
            continue
        if not pointers:
            continue
        m = re.match(r"^s_load_dword(?:x(\d+))?\s+[^,]+,\s*s\[(\d+):\d+\],\s*(0x[0-9a-f]+|\d+)$", text)
        if m and int(m.group(2)) in pointers:
            end = int(m.group(3), 0) + 4 * int(m.group(1) or 1)
            if end > sizes[kernel]:
                bad.append(f"{kernel}: {text} reads to {end} of {sizes[kernel]} bytes of arguments")
        copy = re.match(r"^s_mov_b64\s+s\[(\d+):\d+\],\s*s\[(\d+):\d+\]$", text)
        copied = bool(copy) and int(copy.group(2)) in pointers
        m = re.match(r"^(?:s_(?!cmp|bitcmp|store|waitcnt|cbranch|branch)\w+|v_read\w+)\s+s(?:(\d+)|\[(\d+):(\d+)\])", text)
        if m:  # what is written over is a pointer no longer
            lo, hi = (int(m.group(1)),) * 2 if m.group(1) else (int(m.group(2)), int(m.group(3)))
            pointers -= set(range(lo - 1, hi + 1))
        if copied:
            pointers.add(int(copy.group(1)))
    return bad


def early_mfma_result_uses(src: str, extra_flags=()) -> list[str]:
    """Compiles `src` to gfx950 assembly and lists every instruction other than an MFMA that touches an ordinary
    register which an assembly MFMA (v_mfma_f32_16x16x32) wrote fewer than eight wait states before. Eight is the distance that the
    compiler keeps behind its own MFMAs of that form (v_mfma, s_nop 7, use); around assembly
    statements it keeps none. Every instruction counts as one state, MFMAs too, which take longer. A branch or
    a label within the distance is listed as well: what follows it is not known here."""
    import re
    states_needed = 8
    vgpr = re.compile(r"\bv(?:(\d+)|\[(\d+):(\d+)\])")

    def registers(text):
        return {r for one, lo, hi in vgpr.findall(text) for r in (range(int(one), int(one) + 1) if one else range(int(lo), int(hi) + 1))}

    bad, kernel, in_asm = [], "", False
    flying = []  # [registers, wait states since, the MFMA]
    for line in _device_asm(src, extra_flags):
        if "#ASMSTART" in line or "#ASMEND" in line:
            in_asm = "#ASMSTART" in line
            continue
        text = line.split(";")[0].strip()
        if not text or (text.startswith(".") and not text.endswith(":")):
            continue
        if text.endswith(":") or re.match(r"^s_(c?branch|setpc|endpgm)", text):
            if not text.startswith((".", "s_")):
                kernel = text[:-1]
            elif not text.startswith("s_endpgm"):
                bad += [f"{kernel}: {mfma} | {states} wait states | {text}" for _, states, mfma in flying]
            flying = []
            continue
        own = re.match(r"^v_mfma_f32_16x16x32\S*\s+(v\[\d+:\d+\])", text) if in_asm else None
        if not text.startswith("v_mfma"):
            bad += [f"{kernel}: {mfma} | {states} wait states | {text}" for regs, states, mfma in flying if regs & registers(text)]
        if own:
            flying = [f for f in flying if not f[0] & registers(own.group(1))]  # the chain's next: waits by itself
        nop = re.match(r"^s_nop\s+(\d+)", text)
        for f in flying:
            f[1] += int(nop.group(1)) + 1 if nop else 1
        flying = [f for f in flying if f[1] < states_needed]
        if own:
            flying.append([registers(own.group(1)), 0, text])
    return bad


def wide_mfma_hazards(extra_flags=()) -> list[str]:
    """The same check for the wide-head kernel (attn_wide.hip, attn_wide_kernel): all of its MFMAs
    are assembly statements, its 256 accumulation registers hold O^T for the whole walk, and every
    step ends with the wait (`s_nop 15` ...) before anything else may read them. Also lists any
    use of scratch memory inside a block that holds such MFMAs: the loop is written to fit the
    register file exactly, and a spill there waits on every load in flight."""
    import re
    src = os.path.join(CSRC, "attn_wide.hip")
    bad = tied_mfma_hazards(src, extra_flags, mfma_prefix="v_mfma_f32_16x16x32", kernel_substr="attn_wide_kernel")
    lines = _device_asm(src, extra_flags)
    kernel, block, mfmas, scratch = "", "", 0, []
    label = re.compile(r"^([.\w$]+):")

    def close():
        if "attn_wide_kernel" in kernel and mfmas >= 32 and scratch:
            bad.append(f"{kernel}: {len(scratch)} scratch accesses in {block} beside {mfmas} MFMAs, e.g. {scratch[0]}")

    for line in lines:
        text = line.split(";")[0].strip()
        if not text:
            continue
        m = label.match(text)
        if m:
            close()
            if not text.startswith("."):
                kernel = m.group(1)
            block, mfmas, scratch = m.group(1), 0, []
            continue
        if text.startswith("v_mfma"):
            mfmas += 1
        elif text.startswith("scratch_"):
            scratch.append(text)
    close()
    return bad


def early_store_data_writes(src: str, extra_flags=()) -> list[str]:
    """Compiles `src` to gfx950 assembly and lists every vector instruction that writes a data register of a store of
    more than 8 bytes per lane fewer than two wait states behind it. The store may still be reading that register; the
    compiler keeps the distance behind its own stores, not behind those that are assembly statements."""
    import re
    lines = [l.split(";")[0].strip() for l in _device_asm(src, extra_flags)]
    lines = [l for l in lines if l and (not l.startswith(".") or l.endswith(":"))]
    vectors = re.compile(r"\bv(?:(\d+)|\[(\d+):(\d+)\])")

    def registers(text):
        return {r for one, lo, hi in vectors.findall(text) for r in (range(int(one), int(one) + 1) if one else range(int(lo), int(hi) + 1))}

    bad, kernel = [], ""
    for i, text in enumerate(lines):
        if text.endswith(":") and not text.startswith("."):
            kernel = text[:-1]
        store = re.match(r"^(global|flat|scratch|buffer)_store_dwordx[34]\s+(.*)", text)
        if not store:
            continue
        data, states = registers(store.group(2).split(",")[0 if store.group(1) == "buffer" else 1]), 0
        for later in lines[i + 1:i + 4]:
            if states >= 2:
                break
            # (an exchange of registers writes both of its operands)
            ops = later.split(",")
            if later.startswith("v_") and data & registers(",".join(ops[:2]) if "swap" in ops[0] else ops[0]):
                bad.append(f"{kernel}: {text} | {states} wait states | {later}")
                break
            nop = re.match(r"^s_nop\s+(\d+)", later)
            states += int(nop.group(1)) + 1 if nop else 0 if later.endswith(":") else 1
    return bad


def build_host(verbose: bool = False) -> str:
    os.makedirs(LIBDIR, exist_ok=True)
    srcs = [os.path.join(HOST, f) for f in sorted(os.listdir(HOST)) if f.endswith(".cc")]
    _run(["g++", "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wextra",
          "-I", os.path.join(ROOT, "include"), "-o", HOST_LIB, *srcs,
          "-L", LIBDIR, "-lzdraw_hip", "-Wl,-rpath,$ORIGIN"])
    if verbose:
        print("built", HOST_LIB)
    return HOST_LIB


def check_hand_scheduled_kernels(verbose: bool = False):
    """The GEMM's hand-placed MFMAs and its M0 held across loads are safe only as long as the
    compiler puts nothing of its own in between: a toolchain that does fails the build here."""
    files = [os.path.join(CSRC, f) for f in ("attn_fwd.hip", "attn_wide.hip", "gemm_half.hip", "qk_prepass.hip")]
    from concurrent.futures import ThreadPoolExecutor
    with ThreadPoolExecutor(max_workers=len(files)) as pool:  # one compilation per file, kept for all checks
        list(pool.map(_device_asm, files))
    bad = m0_writes() + m0_writes(files[1], "attn_wide_kernel") + tied_mfma_hazards() + wide_mfma_hazards()
    for f in files:
        bad += vmem_sgpr_hazards(f) + early_store_data_writes(f) + kernarg_overreads(f) + early_mfma_result_uses(f)
    if bad:
        raise RuntimeError("a kernel compiled to code that breaks its hand-written schedule:\n  " + "\n  ".join(bad))
    if verbose:
        print("hand-scheduled kernels: no foreign M0 write, no accumulator touched inside an MFMA run, no load on a scalar register just written, no write of a store's data right behind it, no read past a kernel's arguments, no MFMA result used early")


def build_all(verbose: bool = False):
    build_hip(verbose)
    build_host(verbose)
    check_hand_scheduled_kernels(verbose)


if __name__ == "__main__":
    build_all(verbose=True)
