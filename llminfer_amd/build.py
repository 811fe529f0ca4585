"""Builds libllmi_hip.so (HIP kernels + C ABI) for gfx950 with hipcc, in-tree."""
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB_PATH = os.path.join(HERE, "libllmi_hip.so")
HOST_LIB_PATH = os.path.join(HERE, "libllmi_host.so")
DIAG_LIB_PATH = os.path.join(HERE, "libllmi_diag.so")
TORCH_OPS_PATH = os.path.join(HERE, "_torch_ops.so")

HIP_SOURCES = ["mha_decode_group4.hip", "mha_decode_group8.hip", "mha_decode_group16.hip", "mha_decode_group2.hip", "mha_decode_group1.hip", "mha_stack.hip", "mha_heads.hip",
               "mha_decode.hip", "qk_norm_rope.hip", "gemv.hip", "probes.hip", "c_api.cpp", "pool.cpp"]
DIAG_SOURCES = ["diag_probes.hip"]

# -packed-fp32-ops: keep the compiler from forming packed fp32 VALU ops.
HIPCC_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument",
]


def _run(cmd):
    res = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in res.stdout.splitlines() if "packed-fp32-ops" not in l)
    if res.returncode != 0:
        raise RuntimeError("build failed: %s\n%s" % (" ".join(cmd), out))
    return out


def kernels_using_scratch(compiler_output):
    """Names of the kernels the compiler gave private (scratch) memory, from its resource-usage remarks. None of the
    kernels here may have any: a kernel with a private segment pays for its set-up at every launch, also when the
    path that spilled never runs (an indexed local array in a rarely taken branch cost 0.1 us per decode call)."""
    bad, name = [], None
    for line in compiler_output.splitlines():
        if "remark: Function Name:" in line:
            name = line.split("Function Name:")[1].split("[")[0].strip()
        elif "ScratchSize [bytes/lane]:" in line:
            if int(line.split("ScratchSize [bytes/lane]:")[1].split("[")[0]) != 0:
                bad.append(name)
    return bad


_REGISTERS = re.compile(r"\b(?:s(\d+)\b|s\[(\d+):(\d+)\]|(vcc_lo|vcc_hi|vcc|m0)\b)")
_VMEM = ("global_", "buffer_", "flat_", "scratch_", "tbuffer_")
_WAIT_STATES = 5  # between a vector instruction that writes a scalar register and a memory instruction that reads it


def _scalar_registers(operands):
    regs = set()
    for one, lo, hi, name in _REGISTERS.findall(operands):
        if name:
            regs |= {"vcc_lo", "vcc_hi"} if name == "vcc" else {name}
        else:
            regs |= set(range(int(lo or one), int(hi or one) + 1))
    return regs


def scalar_reads_too_early(disassembly):
    """Memory instructions that read a scalar register fewer than five wait states behind the vector instruction that
    wrote it, as "kernel: writer -> reader", from llvm-objdump's output. The compiler keeps that distance for its own
    instructions and does not look into asm statements, and the LDS-DMA loads are asm statements: with their base in
    vector registers it puts the v_readfirstlane pair right in front of the load, which then goes to a wrong address."""
    found = set()
    for kernel, body in re.findall(r"^[0-9a-f]+ <(\S+)>:\n(.*?)(?=^[0-9a-f]+ <|\Z)", disassembly, re.M | re.S):
        code, index, jumps = [], {}, []
        for line in body.splitlines():
            text, _, where = line.partition("//")
            if not where:
                continue
            name, _, operands = text.strip().partition(" ")
            index[int(where.partition(":")[0], 16)] = len(code)
            if "branch" in name:
                jumps.append((len(code), int(where.rpartition("+0x")[2].rstrip(">") or "0", 16)))
            code.append((name, operands.strip()))
        ends = ("s_branch", "s_endpgm", "s_setpc_b64")
        before = [[i - 1] if i and code[i - 1][0] not in ends else [] for i in range(len(code))]
        first = min(index, default=0)
        for i, target in jumps:
            if first + target in index:
                before[index[first + target]].append(i)

        def look(i, watched, states, reader):
            if states >= _WAIT_STATES or not watched:
                return
            for j in before[i]:
                name, operands = code[j]
                fields = operands.split(", ")
                if name.startswith("v_"):
                    # (the carry of an addition and the scale of a division come second)
                    written = _scalar_registers(fields[0]) | (_scalar_registers(fields[1]) if "_co_" in name or "div_scale" in name else set())
                    if written & watched:
                        found.add("%s: %s %s -> %s %s" % ((kernel, name, operands) + reader))
                        continue
                    left = watched
                elif name.startswith("s_") and not re.match(r"s_(cmp|bitcmp|cbranch|branch|waitcnt|nop|barrier|sleep|setprio)", name):
                    left = watched - _scalar_registers(fields[0])  # (rewritten by the scalar unit: no distance to keep)
                else:
                    left = watched
                look(j, left, states + (int(operands, 0) + 1 if name == "s_nop" else 1), reader)

        for i, (name, operands) in enumerate(code):
            if name.startswith(_VMEM):
                look(i, _scalar_registers(operands) | ({"m0"} if "_lds_" in name or operands.endswith(" lds") else set()), 0, (name, operands))
    return sorted(found)


def _early_scalar_reads(obj):
    """... in the gfx950 code of an object file that was just built, disassembled."""
    import tempfile

    def tool(name, *args):
        return _run([_run([os.environ.get("HIPCC", "hipcc"), "--print-prog-name=" + name]).strip()] + list(args))

    with tempfile.TemporaryDirectory() as tmp:
        bundle, code = os.path.join(tmp, "bundle"), os.path.join(tmp, "code")
        tool("llvm-objcopy", "--dump-section", ".hip_fatbin=" + bundle, obj, os.path.join(tmp, "rest"))
        tool("clang-offload-bundler", "--type=o", "--unbundle", "--targets=hipv4-amdgcn-amd-amdhsa--gfx950", "--input=" + bundle, "--output=" + code)
        listing = tool("llvm-objdump", "-d", code)
    if "s_endpgm" not in listing:
        raise RuntimeError("no gfx950 code found in " + obj)
    return scalar_reads_too_early(listing)


def _compile_objects(sources, defines, tag):
    """Each source to an object file (in parallel: the kernels' file takes minutes, the others seconds), the
    compiler's remarks of all of them joined."""
    from concurrent.futures import ThreadPoolExecutor
    hipcc = os.environ.get("HIPCC", "hipcc")
    obj_dir = os.path.join(HERE, "build", tag)
    os.makedirs(obj_dir, exist_ok=True)
    flags = [f for f in HIPCC_FLAGS if f != "-shared"]

    def one(src):
        obj = os.path.join(obj_dir, os.path.basename(src) + ".o")
        cmd = [hipcc] + flags + ["-c", "-Rpass-analysis=kernel-resource-usage"] + ["-D" + d for d in defines]
        cmd += ["-I" + os.path.join(ROOT, "include"), "-I" + CSRC, src, "-o", obj]
        remarks = _run(cmd)
        early = _early_scalar_reads(obj) if src.endswith(".hip") else []
        if early:
            raise RuntimeError("scalar registers read too early by a memory instruction (pin them, see scalar_bases in mha_device_helpers.h):\n"
                               + "\n".join(early))
        return obj, remarks

    with ThreadPoolExecutor(max_workers=min(8, len(sources))) as pool:
        results = list(pool.map(one, sources))
    return [o for o, _ in results], "\n".join(out for _, out in results)


def _link_shared(objects, output):
    hipcc = os.environ.get("HIPCC", "hipcc")
    _run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objects + ["-o", output])
    return output


def _check_remarks(out, verbose):
    bad = kernels_using_scratch(out)
    if bad:
        raise RuntimeError("kernels with a private (scratch) segment: %s" % ", ".join(sorted(set(bad))))
    # (the remarks themselves are not worth printing: a dozen lines for each of a hundred kernels)
    out = "\n".join(l for l in out.splitlines() if "-Rpass-analysis" not in l and not re.match(r"^\s*\d*\s*\|", l)
                    and not l.startswith("In file included from"))
    if verbose and out.strip():
        print(out)


def build_hip_library(verbose=False, defines=(), output=None, only=()):
    """`defines`: extra NAME=VALUE macros (the kernels' build-time switches, e.g. LLMI_PV_VALU=1);
    `output`: where to write a variant build instead of the in-tree library; `only`: the sources the defines
    matter to (the others are taken from the in-tree build's objects, which must exist)."""
    tag = "hip" if not (defines or output) else "variant_" + re.sub(r"[^A-Za-z0-9_.-]", "_", os.path.basename(output or "x"))
    sources = [s for s in HIP_SOURCES if not only or s in only]
    objects, out = _compile_objects([os.path.join(CSRC, s) for s in sources], list(defines), tag)
    _check_remarks(out, verbose)
    objects += [os.path.join(HERE, "build", "hip", s + ".o") for s in HIP_SOURCES if s not in sources]
    return _link_shared(objects, output or LIB_PATH)


def build_diag_library(verbose=False):
    """libllmi_diag.so: the two diagnostic probes (include/llmi_hip_diag.h), a library of their own."""
    objects, out = _compile_objects([os.path.join(CSRC, "diag", s) for s in DIAG_SOURCES], [], "diag")
    _check_remarks(out, verbose)
    return _link_shared(objects, DIAG_LIB_PATH)


def build_host_library(verbose=False):
    """The C++17 mirror of the reference's tensor/op/registry interface, linked against libllmi_hip.so."""
    host_dir = os.path.join(CSRC, "host")
    if not os.path.isdir(host_dir):
        return None
    srcs = sorted(os.path.join(host_dir, f) for f in os.listdir(host_dir) if f.endswith(".cpp"))
    hipcc = os.environ.get("HIPCC", "hipcc")
    cmd = [hipcc, "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-Wno-unused-command-line-argument",
           "-I" + os.path.join(ROOT, "include"), "-I" + host_dir] + srcs
    cmd += ["-L" + HERE, "-lllmi_hip", "-Wl,-rpath,$ORIGIN", "-o", HOST_LIB_PATH]
    out = _run(cmd)
    if verbose and out.strip():
        print(out)
    return HOST_LIB_PATH


def build_torch_ops(verbose=False):
    """_torch_ops.so: the native calls of llminfer_amd.ops (a CPython extension against the installed torch; no device code)."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    src = os.path.join(CSRC, "front", "torch_ops.cpp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-Wall", "-fvisibility=hidden",
           "-D_GLIBCXX_USE_CXX11_ABI=%d" % int(torch._C._GLIBCXX_USE_CXX11_ABI), "-I" + os.path.join(ROOT, "include")]
    for d in cpp_extension.include_paths() + [sysconfig.get_paths()["include"]]:
        cmd += ["-isystem", d]
    cmd += [src, "-L" + os.path.join(os.path.dirname(torch.__file__), "lib"), "-ltorch_python", "-ltorch_cpu", "-lc10", "-o", TORCH_OPS_PATH]
    out = _run(cmd)
    if verbose and out.strip():
        print(out)
    return TORCH_OPS_PATH


def build_all(verbose=False):
    paths = [build_hip_library(verbose), build_diag_library(verbose), build_torch_ops(verbose)]
    host = build_host_library(verbose)
    if host:
        paths.append(host)
    return paths


if __name__ == "__main__":
    import argparse
    ap = argparse.ArgumentParser(description="Builds the gfx950 library and the host layer in-tree, or a variant of the library.")
    ap.add_argument("--define", action="append", default=[], metavar="NAME=VALUE",
                    help="build-time switch of the kernels (LLMI_PV_VALU=1, LLMI_STAGES=3, ...); needs --output")
    ap.add_argument("--output", default=None, help="write a variant of libllmi_hip.so here (load it with LLMI_HIP_LIBRARY)")
    ap.add_argument("--only", action="append", default=[], metavar="SOURCE",
                    help="recompile only this source (e.g. mha_stack.hip) for the variant; the rest comes from the in-tree build")
    cli = ap.parse_args()
    if cli.define or cli.output:
        if not cli.output:
            ap.error("--define needs --output: the in-tree library is always the default build")
        print("built", build_hip_library(verbose=True, defines=cli.define, output=os.path.abspath(cli.output), only=cli.only))
        sys.exit(0)
    for p in build_all(verbose=True):
        print("built", p)
    sys.exit(0)
