"""Build libeagle_mi355x.so (the C-ABI library) in-tree with hipcc for gfx950.

    python -m mlx_eagle_spec_decoding_tree_amd.build        # or build.build()

hipcc cross-compiles without a GPU.  Packed fp32 instructions are disabled for
all device code (-packed-fp32-ops).

The compile also asks the backend for every kernel's resource usage
(-Rpass-analysis=kernel-resource-usage) and fails if a kernel that is not on
the list below keeps registers in scratch memory: a spill in a kernel of the
verification step or of the draft loop is a build error, not a slow surprise.
"""
import glob
import os
import re
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libeagle_mi355x.so")
HOST = os.path.join(HERE, "_host.so")

FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    "-fvisibility=hidden", "-fno-gpu-rdc",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument",
    "-Rpass-analysis=kernel-resource-usage",
]

# Kernels that may spill, by a pattern on the demangled-free (mangled) name, with the reason.
# None of them runs in the verification step or in the draft loop of the benchmark configurations.
SCRATCH_ALLOWED = [
    # prompt chunks of 256 x rows by 256 weight rows: 256 accumulator registers, and the addresses of the epilogue
    # kept around the loop (nothing is stored or read inside it); 128 x 256 with scales a group or two at a time
    (r"qmm_gemm_w4g64_kernelILi2ELi[48]E", "prompt GEMM, 256-column blocks"),
    # sixteen waves (K above 3072) leave a wave 128 registers: too few with a second weight tile
    # (SwiGLU, rope) or with the norm weights of three chunks; the drafter's K is 896 there
    (r"qmm_small_kernelILi1[346]ELi[23]ELi\dELi[12]E", "small-row kernel, sixteen waves, two tiles"),
    (r"qmm_small_kernelILi1[36]ELi3ELi\dELi0ELb1E", "small-row kernel, sixteen waves, norm folded in"),
]

_NAME = re.compile(r"Function Name: (\S+)")
_SCRATCH = re.compile(r"ScratchSize \[bytes/lane\]: (\d+)")


def scratch_report(text):
    """{kernel name: scratch bytes per lane} from the resource-usage remarks of one compile."""
    out = {}
    name = None
    for line in text.splitlines():
        m = _NAME.search(line)
        if m:
            name = m.group(1)
            continue
        m = _SCRATCH.search(line)
        if m and name:
            out[name] = int(m.group(1))
            name = None
    return out


def check_scratch(report):
    """Raise if a kernel outside SCRATCH_ALLOWED spills; returns the allowed ones that do."""
    allowed, bad = {}, {}
    for name, nbytes in report.items():
        if nbytes == 0:
            continue
        why = next((w for pat, w in SCRATCH_ALLOWED if re.search(pat, name)), None)
        (allowed if why else bad)[name] = (nbytes, why)
    if bad:
        lines = "\n".join(f"  {n}: {b} bytes per lane" for n, (b, _) in sorted(bad.items()))
        raise RuntimeError("kernels with registers spilled to scratch memory:\n" + lines)
    return allowed


def hipcc():
    for cand in (shutil.which("hipcc"), "/opt/rocm/bin/hipcc"):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found; the HIP extension cannot be built")


def sources():
    return sorted(glob.glob(os.path.join(CSRC, "*.hip")))


def start_host(objdir):
    """Start the compiles of csrc/*.cpp, the native host path of the operators (no device code): a
    Python module on torch's C++ interface.  Returns [(source, object, process)]."""
    import sysconfig
    import torch
    from torch.utils import cpp_extension
    out = []
    for src in sorted(glob.glob(os.path.join(CSRC, "*.cpp"))):
        obj = os.path.join(objdir, os.path.basename(src) + ".o")
        cmd = ["g++", "-O2", "-std=c++17", "-fPIC", "-fvisibility=hidden", "-w", "-D__HIP_PLATFORM_AMD__=1", "-DUSE_ROCM=1",
               f"-D_GLIBCXX_USE_CXX11_ABI={int(torch._C._GLIBCXX_USE_CXX11_ABI)}",
               *(f"-isystem{d}" for d in cpp_extension.include_paths()), "-isystem/opt/rocm/include",
               f"-isystem{sysconfig.get_paths()['include']}", "-c", src, "-o", obj]
        out.append((src, obj, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
    return out


def link_host(compiles):
    from torch.utils import cpp_extension
    objs = []
    for src, obj, p in compiles:
        out, _ = p.communicate()
        if p.returncode != 0:
            raise RuntimeError(f"g++ failed on {src}:\n" + out.decode(errors="replace"))
        objs.append(obj)
    libs = cpp_extension.library_paths()
    tmp = HOST + ".tmp"
    cmd = ["g++", "-shared", *objs, "-o", tmp, *(f"-L{d}" for d in libs), "-L/opt/rocm/lib", f"-L{HERE}",
           "-l:libeagle_mi355x.so", "-ltorch_python", "-ltorch", "-ltorch_cpu", "-ltorch_hip", "-lc10", "-lc10_hip",
           "-lamdhip64", "-Wl,-rpath,$ORIGIN"]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    if r.returncode != 0:
        raise RuntimeError("link of the host module failed:\n" + r.stdout.decode(errors="replace"))
    os.replace(tmp, HOST)


def run_all(cmds, logs, jobs):
    """Run the commands, at most `jobs` at once, and return (return code, what it printed) of each.  They print into files: more
    than a pipe holds would stop a command while another one is waited for."""
    procs = []
    for cmd, path in zip(cmds, logs):
        running = [p for p in procs if p.poll() is None]
        if len(running) >= jobs:
            running[0].wait()
        with open(path, "wb") as log:
            procs.append(subprocess.Popen(cmd, stdout=log, stderr=subprocess.STDOUT))
    out = []
    for p, path in zip(procs, logs):
        p.wait()
        with open(path, "rb") as log:
            out.append((p.returncode, log.read().decode(errors="replace")))
    return out


def build(verbose=False, jobs=8):
    """Compile every csrc/*.hip to an object (in parallel) and link the library, then the host
    module on top of it."""
    cc = hipcc()
    objdir = os.path.join(HERE, "build")
    os.makedirs(objdir, exist_ok=True)
    host = start_host(objdir)
    flags = [f for f in FLAGS if f != "-shared"]
    objs = [os.path.join(objdir, os.path.basename(src) + ".o") for src in sources()]
    cmds = [[cc, *flags, "-c", src, "-o", obj] for src, obj in zip(sources(), objs)]
    if verbose:
        print("\n".join(" ".join(cmd) for cmd in cmds))
    report = {}
    for src, (code, text) in zip(sources(), run_all(cmds, [obj + ".log" for obj in objs], jobs)):
        report.update(scratch_report(text))
        noise = ("is not a recognized feature for this target", "-Rpass-analysis=kernel-resource-usage")
        text = "\n".join(l for l in text.splitlines() if not any(n in l for n in noise))
        if code != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{text}")
        if verbose and text.strip():
            print(text)
    if not report:
        raise RuntimeError("the compiler reported no kernel resource usage: the scratch check cannot run")
    allowed = check_scratch(report)
    if verbose:
        print(f"[build] {len(report)} kernels, {len(allowed)} on the allowed list use scratch memory")
        for n, (b, why) in sorted(allowed.items()):
            print(f"[build]   {b:4d} B/lane  {why}: {n}")
    tmp = LIB + ".tmp"
    cmd = [cc, "--offload-arch=gfx950", "-shared", "-fPIC", "-fno-gpu-rdc", *objs, "-o", tmp]
    r = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)
    if r.returncode != 0:
        raise RuntimeError("link failed:\n" + r.stdout.decode(errors="replace"))
    os.replace(tmp, LIB)
    link_host(host)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
