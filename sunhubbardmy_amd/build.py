"""Build libsunhip.so in-tree for gfx950 with hipcc (no JIT, no torch extension machinery)."""
import os
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libsunhip.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # packed FP32 instructions stay disabled in every device pass of this project
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]


def hipcc():
    rocm = os.environ.get("ROCM_PATH", "/opt/rocm")
    return os.path.join(rocm, "bin", "hipcc")


# translation units, compiled side by side: source and its own definitions
UNITS = [("sunhip.hip", []), ("fft_kernels.hip", []), ("factor.hip", []), ("stock_kernels.hip", [])] + [
    ("update_kernels.hip", ["-DUPD_WHOLE=%d" % w, "-DUPD_NF=%d" % f]) for w in (0, 1) for f in (0, 2)]


def build(verbose=False):
    objs = [os.path.join(CSRC, "unit%d.o" % k) for k in range(len(UNITS))]
    cmds = [[hipcc()] + HIPCC_FLAGS + defs + ["-c", os.path.join(CSRC, s), "-o", o] for (s, defs), o in zip(UNITS, objs)]
    procs = []
    for cmd in cmds:
        if verbose:
            print(" ".join(cmd), flush=True)
        procs.append(subprocess.Popen(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True))
    out = [p.communicate()[0] for p in procs]
    link = [hipcc(), "--offload-arch=gfx950", "-fPIC", "-shared"] + objs + ["-o", OUT + ".tmp"]
    if any(p.returncode for p in procs):
        sys.stderr.write("".join(out))
        raise RuntimeError("hipcc failed building libsunhip.so")
    res = subprocess.run(link, capture_output=True, text=True)
    if res.returncode != 0:
        sys.stderr.write(res.stdout + res.stderr)
        raise RuntimeError("hipcc failed linking libsunhip.so")
    os.replace(OUT + ".tmp", OUT)
    for o in objs:
        os.remove(o)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
