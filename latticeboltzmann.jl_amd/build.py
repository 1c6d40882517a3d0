"""Build liblbm_hip.so for gfx950 with hipcc (no GPU needed to compile).

    python latticeboltzmann.jl_amd/build.py          # incremental
    python latticeboltzmann.jl_amd/build.py --force  # rebuild everything

Translation units and their floating-point contracts:

* ``k_*f64*.hip``, ``kernels_aux.hip``, ``lbm_capi.cpp``, ``lbm_dispatch.cpp``:
  ``-ffp-contract=off`` -- every multiply and add rounds separately, the
  reference's Julia semantics, so the FP64 path reproduces the CPU restatement
  bit for bit;
* ``k_{f32,f16dev,bf16dev}_*.hip``: reduced-precision storages with FP32
  arithmetic, ``-ffp-contract=fast``.

One translation unit per (storage, quadrature group) keeps each hipcc job
small; they compile in parallel.

All device code is built with packed FP32 instructions disabled
(``-target-feature -packed-fp32-ops``).
"""
from __future__ import annotations

import argparse
import os
import shutil
import subprocess
import sys
import tempfile
import time

HERE = os.path.dirname(os.path.abspath(__file__))
REPO = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
BUILD = os.path.join(HERE, "_build")
LIBDIR = os.path.join(HERE, "lib")
LIB = os.path.join(LIBDIR, "liblbm_hip.so")
ARCH = os.environ.get("LBM_OFFLOAD_ARCH", "gfx950")

HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

COMMON = [
    f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-function", "-Wno-unused-variable",
    f"-I{os.path.join(REPO, 'include')}", f"-I{CSRC}",
]

def _units():
    units = [("kernels_aux.hip", ["-ffp-contract=off"]),
             ("lbm_capi.cpp", ["-x", "hip", "-ffp-contract=off"]),
             ("lbm_dispatch.cpp", ["-x", "hip", "-ffp-contract=off"])]
    for name in sorted(os.listdir(CSRC)):
        if name.startswith("k_") and name.endswith(".hip"):
            contract = "off" if "_f64" in name else "fast"
            units.append((name, [f"-ffp-contract={contract}"]))
    return units

def _deps(src):
    """Headers a unit includes (directly or through lbm_kernels.h)."""
    kern = [os.path.join(CSRC, h) for h in ("lbm_quad.h", "lbm_internal.h", "lbm_kernels.h")]
    if src == "lbm_capi.cpp":
        return [os.path.join(CSRC, "lbm_internal.h"), os.path.join(CSRC, "lbm_quad.h"),
                os.path.join(REPO, "include", "lbm_hip.h")]
    if src == "lbm_dispatch.cpp":
        return [os.path.join(CSRC, "lbm_internal.h")]
    if src.startswith("k_multi"):
        return kern + [os.path.join(CSRC, "lbm_multi.h")]
    if src.startswith("k_stage"):
        return kern + [os.path.join(CSRC, "lbm_multi.h"), os.path.join(CSRC, "lbm_stage.h")]
    if src.startswith("k_adjoint"):
        return kern + [os.path.join(CSRC, "lbm_multi.h"), os.path.join(CSRC, "lbm_adjoint.h")]
    return kern


def _mtime(p):
    return os.path.getmtime(p) if os.path.exists(p) else -1.0


def build(force: bool = False, verbose: bool = False) -> str:
    os.makedirs(BUILD, exist_ok=True)
    os.makedirs(LIBDIR, exist_ok=True)
    jobs = []
    objs = []
    for src, flags in _units():
        s = os.path.join(CSRC, src)
        o = os.path.join(BUILD, src.rsplit(".", 1)[0] + ".o")
        objs.append(o)
        newest_dep = max(_mtime(d) for d in _deps(src))
        if not force and _mtime(o) >= max(_mtime(s), newest_dep):
            continue
        jobs.append((src, [HIPCC, *COMMON, *flags, "-c", s, "-o", o]))
    # heaviest units first, at most one hipcc per CPU
    jobs.sort(key=lambda j: (not j[0].startswith("k_"),
                             "q37" not in j[0] and "multi_f" not in j[0]
                             and "stage" not in j[0], j[0]))
    width = max(1, min(len(jobs), os.cpu_count() or 1, 16))
    procs = []
    failed = []
    pending = list(jobs)
    while pending or procs:
        while pending and len(procs) < width:
            src, cmd = pending.pop(0)
            if verbose:
                print(" ".join(cmd), flush=True)
            log = tempfile.TemporaryFile()
            procs.append((src, subprocess.Popen(cmd, stdout=log, stderr=subprocess.STDOUT), log))
        time.sleep(0.05)
        done = [q for q in procs if q[1].poll() is not None]
        if not done:
            continue
        procs.remove(done[0])
        src, p, log = done[0]
        log.seek(0)
        text = log.read().decode(errors="replace")
        log.close()
        # the host pass does not know the packed-fp32 target feature; that warning is harmless
        lines = [ln for ln in text.splitlines() if "packed-fp32-ops" not in ln
                 and "not a recognized feature" not in ln]
        if p.returncode != 0:
            failed.append(src)
            print("\n".join(lines), file=sys.stderr)
        elif verbose and lines:
            print("\n".join(lines))
    if failed:
        raise RuntimeError(f"hipcc failed for {failed}")
    if force or procs or not os.path.exists(LIB) or _mtime(LIB) < max(_mtime(o) for o in objs):
        tmp = LIB + ".tmp"
        cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", *objs, "-o", tmp]
        if verbose:
            print(" ".join(cmd), flush=True)
        subprocess.run(cmd, check=True)
        os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    ap = argparse.ArgumentParser()
    ap.add_argument("--force", action="store_true")
    ap.add_argument("-v", "--verbose", action="store_true")
    a = ap.parse_args()
    print(build(force=a.force, verbose=a.verbose))
