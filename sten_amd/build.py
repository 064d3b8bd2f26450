"""Build recipe for libnmg_hip.so (hipcc, gfx950 only) and the host path.  Run as ``python -m sten_amd.build``."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libnmg_hip.so")
SOURCES = ["nmg_runtime.hip", "nmg_sparsify.hip", "nmg_match_f32.hip", "nmg_match_f16.hip", "nmg_match_bf16.hip", "nmg_match_fixed.hip",
           "nmg_spmm.hip", "nmg_smfmac.hip", "nmg_dense.hip", "nmg_split3.hip",
           "nmg_densefrag.hip", "nmg_w4.hip", "nmg_pack.hip", "nmg_sddmm.hip", "nmg_perfect.hip", "nmg_gstream.hip", "nmg_sstream.hip", "nmg_ostream.hip", "nmg_align.hip"]
# bench.py's measurement aid: a library of its own, outside the product ABI
PROBE_LIB = os.path.join(HERE, "libnmg_probe.so")
PROBE_SOURCES = ["nmg_probe.hip"]
# the native host path: an extension module against torch's libraries, linked to LIB
HOST_LIB = os.path.join(HERE, "_host.so")
HOST_SOURCE = "nmg_host.cpp"
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-ffp-contract=off",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]
# Compressor, any group size: with the register usage of match_partial known to its callers the function saves nothing and they spill what it
# touches, up to 500 reads of spilled scalars behind the call.  us, whole blocks, fp16, known -> not: 3:8:8 79 -> 66, 5:8:17 124 -> 104,
# 2:4:64 28.8 -> 26.1, 1025 to 2560 columns 0.9 of the time; the kernels of fixed group sizes lose, 4:8:32 118 -> 125, 2:4:16 59.0 -> 59.7, and keep it.
OPTIONS = {src: ["-mllvm", "-enable-ipra=0"] for src in ("nmg_match_f32.hip", "nmg_match_f16.hip", "nmg_match_bf16.hip")}


def build_host(verbose=False):
    """Compile the host path (no device code) and link it against torch and the library beside it."""
    import sysconfig

    from torch.utils.cpp_extension import include_paths, library_paths
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-fPIC", "-shared", "-D__HIP_PLATFORM_AMD__=1",
           "-I" + sysconfig.get_paths()["include"]]
    cmd += ["-isystem" + p for p in include_paths() + ["/opt/rocm/include"]]
    cmd += [os.path.join(CSRC, HOST_SOURCE), "-o", HOST_LIB, "-L" + HERE, "-l:" + os.path.basename(LIB), "-Wl,-rpath,$ORIGIN"]
    cmd += ["-L" + p for p in library_paths()] + ["-ltorch_python", "-ltorch", "-ltorch_cpu", "-lc10", "-lc10_hip"]
    if verbose:
        print(" ".join(cmd), file=sys.stderr)
    subprocess.run(cmd, check=True)
    return HOST_LIB


def build(verbose=False, jobs=8, check=True):
    """Compile every HIP source for gfx950 and link the shared library in-tree.  With ``check`` the
    compiled kernels that track their loads by hand are re-read (``isa_check``): a register touched
    while its load is in flight fails the build."""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
    objdir = os.path.join(HERE, "_obj")
    os.makedirs(objdir, exist_ok=True)
    procs = []
    objs = []
    for src in SOURCES + PROBE_SOURCES:
        obj = os.path.join(objdir, src.replace(".hip", ".o"))
        if src in SOURCES:
            objs.append(obj)
        cmd = [hipcc] + FLAGS + OPTIONS.get(src, []) + ["-c", os.path.join(CSRC, src), "-o", obj]
        if verbose:
            print(" ".join(cmd), file=sys.stderr)
        procs.append((src, subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT)))
        if len(procs) >= jobs:
            _drain(procs)
    _drain(procs)
    cmd = [hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + objs + ["-o", LIB]
    subprocess.run(cmd, check=True)
    probe_objs = [os.path.join(objdir, src.replace(".hip", ".o")) for src in PROBE_SOURCES]
    subprocess.run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC"] + probe_objs + ["-o", PROBE_LIB], check=True)
    build_host(verbose)
    if check:
        from . import isa_check
        if isa_check.main([]) != 0:
            raise RuntimeError("isa_check: a kernel touches a register whose load is still in flight (see above)")
    return LIB


def _drain(procs):
    while procs:
        src, p = procs.pop(0)
        out, _ = p.communicate()
        text = out.decode(errors="replace")
        # the host pass does not know the packed-fp32 target feature; that note is harmless
        text = "\n".join(l for l in text.splitlines() if "packed-fp32-ops" not in l)
        if p.returncode != 0:
            raise RuntimeError(f"hipcc failed on {src}:\n{text}")
        if text.strip():
            print(text, file=sys.stderr)


if __name__ == "__main__":
    print(build(verbose=True))
