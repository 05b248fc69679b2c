"""Builds libxcquad.so (the HIP library) in place with hipcc for gfx950.

    python -m pdynamo3_amd.build        (or build() from Python)

The library is written next to this file; it is git-ignored and travels with the source tree.
"""

import concurrent.futures
import os
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIBRARY = os.path.join(HERE, "libxcquad.so")
SOURCES = ["xq_alloc.hip", "xq_api.hip", "xq_grid.hip", "xq_basis.hip", "xq_integrate.hip", "xq_f64.hip", "xq_mixed.hip",
           "xq_gradients.hip", "xq_uks.hip", "xq_noalloc.hip", "qs_integrals.hip",
           "qs_fit_low.hip", "qs_fit_dp.hip", "qs_fit_dd_sp.hip", "qs_fit_dd_d.hip", "qs_dense.hip"]
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
FLAGS = ["-O3", "-std=c++17", "-fPIC", "--offload-arch=gfx950",
         # Packed FP32 instructions stay off: hipcc would otherwise form v_pk_* FP32 ops from plain float code.
         "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
         "-Wno-unused-result"]
# rocBLAS and rocSOLVER for the SCF's dense steps (qs_dense.hip).
LIBS = ["-L/opt/rocm/lib", "-lrocsolver", "-lrocblas", "-Wl,-rpath,/opt/rocm/lib"]


def _run(cmd, verbose):
    if verbose:
        print(" ".join(cmd), flush=True)
    subprocess.run(cmd, check=True)


def build(verbose=False):
    """Compile every HIP source, several at a time, and link libxcquad.so; raises CalledProcessError on a compiler error."""
    with tempfile.TemporaryDirectory() as objects:
        def compiled(source):
            out = os.path.join(objects, source + ".o")
            _run([HIPCC] + FLAGS + ["-c", os.path.join(CSRC, source), "-o", out], verbose)
            return out
        # The files of the largest unrolled kernels first: they take the longest.
        slow = sorted(SOURCES, key=lambda s: not s.startswith("qs_fit_"))
        with concurrent.futures.ThreadPoolExecutor(min(8, os.cpu_count() or 1)) as pool:
            files = list(pool.map(compiled, slow))
        _run([HIPCC, "-shared", "-fPIC", "--offload-arch=gfx950", "-o", LIBRARY + ".tmp"] + files + LIBS, verbose)
    os.replace(LIBRARY + ".tmp", LIBRARY)
    return LIBRARY


if __name__ == "__main__":
    build(verbose="-v" in sys.argv)
    print(LIBRARY)
