"""Builds libmhffn_hip.so (the C-ABI library) in-tree with hipcc for gfx950, and the torch extension module over it.

    python -m flashmhf_amd.build

One code object, one architecture; no CUDA headers, no torch headers, links only libamdhip64.  Beside it _native.so, the torch
operators' host side on top of that C ABI (g++, torch's headers).
"""
import os
import re
import subprocess
import sys
import tempfile
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBDIR = os.path.join(HERE, "_lib")
LIB = os.path.join(LIBDIR, "libmhffn_hip.so")
SOURCES = ["mhffn_capi.hip", "mhffn_fwd.hip", "mhffn_bwd.hip", "mhffn_f32.hip", "mhffn_gate.hip", "mhffn_rope.hip", "mhffn_product.hip"]
# those that read LDS from inline assembly and wait by count (reads_touched_in_flight)
ASYNC_READ_SOURCES = ["mhffn_bwd.hip", "mhffn_fwd.hip", "mhffn_product.hip"]
# the torch side: an extension module on top of the C ABI, plain C++
NATIVE_LIB = os.path.join(LIBDIR, "_native.so")
NATIVE_SOURCE = "mhffn_torch.cpp"
# benchmark-only object: a register-resident matrix-instruction loop bench.py times beside the kernels
PROBE_LIB = os.path.join(LIBDIR, "libmhffn_probe.so")
PROBE_SOURCE = "mhffn_probe.hip"
FLAGS = [
    "-O3", "--offload-arch=gfx950", "-fPIC", "-std=c++17",
    # packed fp32 VALU ops are kept out of the generated code on this hardware pool
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
]

# The backward's loops start on a 64-byte line.  Its kernels issue from one or two waves per SIMD, and where the loops fell by chance
# cost dK/dU/dV up to 1.8 % (us as they fell / on a line: 2,048 tokens of 8 heads of 64 with 12 experts of 320 64.4 / 63.5, 16,384 of 8 heads of 128 with 11
# of 352 693 / 689) and dQ/dR up to 1 % (4,096 tokens of 8 heads of 96 76.7 / 76.0).  The forward's gain and lose by it (338 instead of 341, but 43.2
# instead of 42.0 with heads of 64).
SOURCE_FLAGS = {"mhffn_bwd.hip": ["-falign-loops=64"]}


def build_lib(verbose=False, jobs=8):
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    os.makedirs(LIBDIR, exist_ok=True)
    objdir = os.path.join(LIBDIR, "obj")
    os.makedirs(objdir, exist_ok=True)

    usage, touched = {}, {}

    def compile_one(src):
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        cmd = [hipcc, *FLAGS, *SOURCE_FLAGS.get(src, []), "-Rpass-analysis=kernel-resource-usage", "-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, stderr=subprocess.PIPE, text=True)
        # everything the compiler said except the resource-usage remarks and the host pass's note on the packed-fp32
        # feature: a warning keeps its source line and caret
        other = [ln for ln in r.stderr.splitlines() if "packed-fp32-ops" not in ln and "-Rpass-analysis" not in ln]
        if other and (r.returncode or any("warning" in ln or "error" in ln for ln in other)):
            print("\n".join(other), file=sys.stderr, flush=True)
        if r.returncode:
            raise subprocess.CalledProcessError(r.returncode, cmd)
        usage.update(parse_resource_usage(r.stderr))
        return obj

    def check_assembly(src):
        with tempfile.TemporaryDirectory() as tmp:
            out = os.path.join(tmp, "kernels.s")
            subprocess.check_call([hipcc, *FLAGS, *SOURCE_FLAGS.get(src, []), "--offload-device-only", "-S", os.path.join(CSRC, src), "-o", out],
                                  stderr=subprocess.DEVNULL)
            with open(out) as f:
                lines = f.readlines()
        if not any("ds_read" in line for line in lines):
            raise RuntimeError(f"no LDS reads found in the assembly of {src}")
        touched.update(reads_touched_in_flight(lines))

    native_obj = os.path.join(objdir, NATIVE_SOURCE.replace(".cpp", ".o"))
    with ThreadPoolExecutor(max_workers=jobs) as ex:
        native = ex.submit(subprocess.check_call, native_compile(native_obj))
        checks = [ex.submit(check_assembly, src) for src in ASYNC_READ_SOURCES]
        objs = list(ex.map(compile_one, SOURCES + [PROBE_SOURCE]))
        native.result()
        for check in checks:
            check.result()
    for out, members in ((LIB, objs[:-1]), (PROBE_LIB, objs[-1:])):
        cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", out, *members]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.check_call(cmd)
    subprocess.check_call(native_link(native_obj))
    with open(os.path.join(LIBDIR, "resource_usage.txt"), "w") as f:     # registers, scratch, occupancy per kernel
        for name in sorted(usage):
            f.write(name + "  " + "  ".join(f"{k}={v}" for k, v in usage[name].items()) + "\n")
    check_no_scratch(usage)
    check_variants(usage)
    if touched:
        raise RuntimeError(f"registers used before the LDS read that fills them has returned: {touched}")
    return LIB


def native_compile(obj):
    """g++ line of the extension module's one source: torch's, Python's and HIP's headers."""
    import sysconfig
    import torch
    t = os.path.join(os.path.dirname(torch.__file__), "include")
    inc = [t, os.path.join(t, "torch", "csrc", "api", "include"), "/opt/rocm/include", sysconfig.get_paths()["include"]]
    return [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
            f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}", "-Wno-attributes",
            *(f"-isystem{i}" for i in inc), "-c", os.path.join(CSRC, NATIVE_SOURCE), "-o", obj]


def native_link(obj):
    """... and of its link: torch's libraries, libmhffn_hip.so beside it."""
    import torch
    t = os.path.join(os.path.dirname(torch.__file__), "lib")
    return [os.environ.get("CXX", "g++"), "-shared", obj, "-o", NATIVE_LIB, "-L" + LIBDIR, "-lmhffn_hip", "-L" + t, "-lc10",
            "-lc10_hip", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-ltorch_python", "-Wl,-rpath,$ORIGIN"]


def parse_resource_usage(stderr_text):
    """{kernel symbol: {field: value}} from hipcc's -Rpass-analysis=kernel-resource-usage remarks."""
    usage, cur = {}, None
    for line in stderr_text.splitlines():
        m = re.search(r"remark:\s+Function Name: (\S+)", line)
        if m:
            cur = usage.setdefault(m.group(1), {})
            continue
        m = re.search(r"remark:\s+([A-Za-z ]+?)(?: \[[^\]]*\])?: (\S+) \[-Rpass", line)
        if m and cur is not None:
            cur[m.group(1).strip()] = m.group(2)
    return usage


# Kernels whose code assumes that every value stays in registers, as (name fragment, instantiations expected).
EXPECTED_KERNELS = (
    ("mhffn_fwd_kernel", 3), ("mhffn_bwd_dqdr_kernel", 3), ("mhffn_bwd_dkdudv_kernel", 6),
    ("mhffn_gate_fwd_kernel", 12), ("mhffn_gate_bwd_kernel", 12),
)
# Variants of those kernels for smaller problems and for float32, and the products, under the same rule.  (The prologue's kernels that move
# whole rows and the dK/dU/dV kernels with two waves a block are told by the mode, a type, that their names end in, and are not counted
# among the instantiations above.)
MODES = ("WholeRows", "TokenHalves")
VARIANT_KERNELS = (("mhffn_fwd_rows128_kernel", 3), ("mhffn_fwd_rows32_kernel", 6), ("mhffn_fwd_rows32_long_kernel", 3), ("mhffn_bwd_dqdr_rows32_kernel", 3),
                   ("fwd_f32_kernelILi", 4), ("dqdr_f32_kernelILi", 4), ("dkdudv_f32_kernelILi", 2), ("dkdudv_split_kernelILi", 3),
                   ("fwd_fp32_kernelILi", 4), ("dqdr_fp32_kernelILi", 4),
                   ("WholeRows", 12), ("TokenHalves", 6),
                   ("mhffn_product_kernel", 10), ("mhffn_product_pair_kernel", 9), ("mhffn_product_split_kernel", 2))
# The one instantiation known to spill: head prologue backward for d_h = 128 with more than 32 experts and RMSNorm
# (<128, 2, true>).  It is correct but slow; the block (MHFFNLayer.heads_and_gate) does not route that case to it.
ALLOWED_SCRATCH = ("mhffn_gate_bwd_kernelILi128ELi2ELb1E",)


def check_no_scratch(usage):
    """The hand-scheduled kernels assume every value stays in registers: a spill would put VALU copies of matrix results
    into places the explicit wait states do not cover, and in the bandwidth-bound head prologue it multiplies the
    run time.  Fails the build if the compiler reports private (scratch) memory for one of them, and also if the
    resource remarks of an expected kernel are missing (a changed remark format must not pass silently)."""
    for frag, count in EXPECTED_KERNELS:
        found = [n for n in usage if frag in n and "ScratchSize" in usage[n] and not any(m in n for m in MODES)]
        if len(found) != count:
            raise RuntimeError(f"expected resource-usage remarks for {count} instantiations of {frag}, found {len(found)}")
    for name, u in usage.items():
        if any(frag in name for frag, _ in EXPECTED_KERNELS) and int(u["ScratchSize"]) != 0:
            if any(a in name for a in ALLOWED_SCRATCH):
                continue
            raise RuntimeError(f"{name} uses {u['ScratchSize']} bytes of scratch per lane: a spill in a hand-scheduled kernel")


def check_variants(usage):
    """check_no_scratch's rule for VARIANT_KERNELS, none of which may spill."""
    for frag, count in VARIANT_KERNELS:
        found = [n for n in usage if frag in n and "ScratchSize" in usage[n]]
        if len(found) != count or any(int(usage[n]["ScratchSize"]) for n in found):
            raise RuntimeError(f"expected {count} instantiations of {frag} without scratch memory, found {found}")


def _registers(operand):
    m = re.match(r"([va])(?:(\d+)|\[(\d+):(\d+)\])$", operand)
    if not m:
        return set()
    lo, hi = (m[2], m[2]) if m[2] else (m[3], m[4])
    return {(m[1], k) for k in range(int(lo), int(hi) + 1)}


def _kernels(assembly):
    """(symbol, [(opcode, operands, text)], {label: index into them}) of every kernel of an assembly listing."""
    name = None
    for line in assembly:
        code = line.split(";")[0].strip()
        if m := re.match(r"(_Z\S+):", line):
            name, code_lines, labels = m[1], [], {}
        elif name and line.startswith(".Lfunc_end"):
            yield name, code_lines, labels
            name = None
        elif name and (m := re.match(r"(\.L\S+):", code)):
            labels[m[1]] = len(code_lines)
        elif name and code and not code.startswith(".") and not code.endswith(":"):
            op, _, rest = code.partition(" ")
            code_lines.append((op, rest.strip(), code))


def reads_touched_in_flight(assembly):
    """{kernel symbol: first such instruction} where an instruction uses a register that an LDS read in front of it, on any way through
    the kernel, is still to fill.  LDS reads issued from inline assembly are waited for by count in inline assembly, too; between the two
    the compiler may copy their registers, which it takes for filled: wrong values, depending on timing."""
    found = {}
    for kernel, code, labels in _kernels(assembly):
        registers = [[_registers(t.strip().split(" ")[0]) for t in rest.split(",")] for _, rest, _ in code]
        touched, seen, ways = set(), set(), [(0, ())]        # a way: where it goes on, the registers of each read in flight
        while ways:
            at, in_flight = ways.pop()
            while at < len(code) and (at, in_flight) not in seen:
                seen.add((at, in_flight))
                if len(seen) > 1000 * (len(code) + 1):
                    raise RuntimeError(f"too many ways through {kernel}")
                op, rest, _ = code[at]
                at += 1
                if op == "s_endpgm":
                    break
                if op == "s_waitcnt":
                    m = re.search(r"lgkmcnt\((\d+)\)", rest)
                    if m:                                    # LDS operations return in order
                        in_flight = in_flight[max(0, len(in_flight) - int(m[1])):]
                elif op == "s_branch":
                    at = labels.get(rest, len(code))
                elif op.startswith("s_cbranch"):
                    ways.append((labels.get(rest, len(code)), in_flight))
                else:
                    used = set().union(*registers[at - 1])
                    if any(r & used for r in in_flight):
                        touched.add(at - 1)
                    if op.startswith("ds_"):
                        in_flight = (*in_flight, frozenset(registers[at - 1][0]) if op.startswith("ds_read") else frozenset())[-64:]
        if touched:
            found[kernel] = code[min(touched)][2]
    return found


if __name__ == "__main__":
    print(build_lib(verbose="-q" not in sys.argv))
