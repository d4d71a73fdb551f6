"""In-tree build of libcannon_hip.so for gfx950 (hipcc, no tracing compiler, no JIT cache)."""
import os
import subprocess
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
OUT = os.path.join(HERE, "libcannon_hip.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

# -ffp-contract=off: no fused multiply-adds, every rounding follows the reference's operation
# order; correctly rounded FP32 divide/sqrt and IEEE denormals; packed-FP32 instructions off.
FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC",
    "-ffp-contract=off", "-fno-fast-math", "-fhip-fp32-correctly-rounded-divide-sqrt",
    "-fno-gpu-flush-denormals-to-zero",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-result",
]
# object name, source, further flags: compiled side by side, then linked
UNITS = [
    ("chp_api", "chp_api.hip", []),
    ("chp_narrow_f32", "chp_narrow_kernels.hip", ["-DCHP_REAL=float"]),
    ("chp_narrow_f64", "chp_narrow_kernels.hip", ["-DCHP_REAL=double"]),
]


def build(verbose=False):
    odir = os.path.join(HERE, "_build")
    os.makedirs(odir, exist_ok=True)

    def run(cmd):
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)

    objs = [os.path.join(odir, name + ".o") for name, _, _ in UNITS]
    with ThreadPoolExecutor(len(UNITS)) as pool:
        list(pool.map(lambda u: run([HIPCC] + FLAGS + u[0][2] + ["-c", "-o", u[1], os.path.join(CSRC, u[0][1])]),
                      zip(UNITS, objs)))
    run([HIPCC, "--offload-arch=gfx950", "-shared", "-fPIC", "-o", OUT + ".tmp"] + objs)
    os.replace(OUT + ".tmp", OUT)
    return OUT


if __name__ == "__main__":
    build(verbose=True)
