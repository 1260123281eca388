"""Builds the gfx950 device library (libfnx_mi355x.so) in-tree with hipcc. No GPU is needed to build."""
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libfnx_mi355x.so")
SOURCES = ["fnx_verify.hip", "fnx_window_types.hip"]
FLAGS = [
    "-O3", "--offload-arch=gfx950", "-std=c++17", "-fPIC",
    "-ffp-contract=off",                       # fused multiply-adds only where the code says fmaf: part of the results' definition
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-mllvm", "-amdgpu-mfma-vgpr-form",       # matrix-core results in the ordinary registers: the kernels here take them up with vector instructions right away
    "-Wall", "-Wno-unused-function", "-Wno-unknown-attributes",
]


def build(verbose=False, extra=()):
    """every source to an object of its own, side by side, then the library"""
    hipcc = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

    def text(out):
        return "\n".join(l for l in out.splitlines() if "packed-fp32-ops" not in l and l.strip())

    with tempfile.TemporaryDirectory() as tmp:
        objs = [os.path.join(tmp, s + ".o") for s in SOURCES]
        cmds = [[hipcc, *FLAGS, *extra, "-c", "-o", o, os.path.join(CSRC, s)] for s, o in zip(SOURCES, objs)]
        if verbose:
            print("\n".join(" ".join(c) for c in cmds), flush=True)
        running = [subprocess.Popen(c, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True) for c in cmds]
        outs = [(p.communicate()[0], p.returncode) for p in running]
        for out, rc in outs:
            if rc != 0:
                raise RuntimeError("hipcc failed:\n" + text(out))
        r = subprocess.run([hipcc, "--offload-arch=gfx950", "-fPIC", "-shared", "-o", LIB, *objs], capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("hipcc failed:\n" + text(r.stdout + r.stderr))
        if verbose:
            print("\n".join(t for t in (text(o) for o, _ in outs) if t))
    return LIB


if __name__ == "__main__":
    print(build(verbose=True, extra=sys.argv[1:]))
