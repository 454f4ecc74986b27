"""Compiles the HIP sources of this package into convlogic_amd/libconvlogic_amd.so for gfx950, and the autograd nodes in front of
it (host code) into convlogic_amd/_nodes.so.

hipcc cross-compiles without a GPU, so this runs in the build container; the built library
travels with the tree.  Usage:  python -m convlogic_amd.build
"""
import os
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
SOURCES = ["clg_api.hip", "conv_binary.hip", "logic_fc.hip", "fc_tree.hip", "packbits.hip", "binarize.hip", "conv_generic.hip", "conv_forward.hip", "conv_small.hip", "conv_pair.hip", "conv_pair_grad.hip", "conv_block.hip", "net_step.hip"]
LIB = os.path.join(PKG, "libconvlogic_amd.so")
NODES = os.path.join(PKG, "_nodes.so")


def hipcc_path():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", "hipcc"):
        if cand and (os.path.sep not in cand or os.path.exists(cand)):
            return cand
    raise RuntimeError("hipcc not found")


def build(verbose=False):
    """Compiles every source to an object of its own (in parallel) and links them: the result is the same library a
    single hipcc invocation over all sources gives, in a third of the time."""
    import concurrent.futures
    import tempfile
    hipcc = hipcc_path()
    flags = ["--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
             "-I" + os.path.join(ROOT, "include"), "-I" + os.path.join(PKG, "csrc")]

    def run(cmd):
        if verbose:
            print(" ".join(cmd))
        res = subprocess.run(cmd, capture_output=True, text=True)
        # the host pass does not know the -packed-fp32-ops target feature and says so; that is harmless
        err = "\n".join(l for l in res.stderr.splitlines() if "packed-fp32-ops" not in l)
        if res.returncode != 0:
            raise RuntimeError("hipcc failed:\n" + err)
        if verbose and err.strip():
            print(err, file=sys.stderr)

    with tempfile.TemporaryDirectory(prefix="clg_build_") as tmp:
        objs = [os.path.join(tmp, s.replace(".hip", ".o")) for s in SOURCES]
        nodes = os.path.join(tmp, "nodes.o")
        with concurrent.futures.ThreadPoolExecutor(max_workers=8) as pool:
            jobs = [pool.submit(run, [*_nodes_compiler(), "-c", os.path.join(PKG, "csrc", "nodes.cpp"), "-o", nodes])]
            jobs += [pool.submit(run, [hipcc, *flags, "-c", os.path.join(PKG, "csrc", s), "-o", o]) for s, o in zip(SOURCES, objs)]
            for j in jobs:
                j.result()
        run([hipcc, "--offload-arch=gfx950", "-shared", "-fPIC", *objs, "-o", LIB])
        run(["g++", "-shared", nodes, "-o", NODES, *_torch_libraries(), "-L" + PKG, "-l:libconvlogic_amd.so", "-Wl,-rpath,$ORIGIN"])
    return LIB


def _nodes_compiler():
    """The autograd nodes are host code against torch's headers."""
    import sysconfig

    from torch.utils import cpp_extension
    includes = [*cpp_extension.include_paths("cuda"), sysconfig.get_paths()["include"]]
    return ["g++", "-std=c++17", "-O2", "-fPIC", "-D__HIP_PLATFORM_AMD__", "-DUSE_ROCM", *(a for d in includes for a in ("-isystem", d)),
            "-I" + os.path.join(ROOT, "include")]


def _torch_libraries():
    from torch.utils import cpp_extension
    return ["-L" + d for d in cpp_extension.library_paths("cuda")] + ["-lc10", "-lc10_hip", "-ltorch_cpu", "-ltorch", "-ltorch_python"]


if __name__ == "__main__":
    print(build(verbose=True))
