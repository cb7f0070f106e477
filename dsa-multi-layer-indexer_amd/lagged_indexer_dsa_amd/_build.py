"""Build libdsa_mli.so (the HIP kernels + C ABI) for gfx950, in-tree.

Run as ``python -m lagged_indexer_dsa_amd._build`` or call :func:`build`.
hipcc cross-compiles without a GPU; the library lands next to this file in
``_lib/`` so it travels with the source tree.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile
from pathlib import Path

PKG_DIR = Path(__file__).resolve().parent
ROOT_DIR = PKG_DIR.parent            # dsa-multi-layer-indexer_amd/
REPO_DIR = ROOT_DIR.parent
CSRC = ROOT_DIR / "csrc"
INCLUDE = REPO_DIR / "include"
LIB_DIR = PKG_DIR / "_lib"
LIB_PATH = LIB_DIR / "libdsa_mli.so"
SOURCES = ["libdsa_mli.hip", "capi.hip", "mla_rows.hip", "prefill.hip", "prefill_logits.hip", "select_rows.hip",
           "quant.hip", "sol.hip"]
ARCH = "gfx950"


def hipcc() -> str:
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and Path(cand).exists():
            return cand
    raise RuntimeError("hipcc not found: the DSA HIP library cannot be built")


def build(verbose: bool = False, out: Path | None = None, phase_stamps: bool = False) -> Path:
    """Compile every HIP source into LIB_PATH, or `out` (always recompiles).
    phase_stamps: compile in the per-phase timestamps (profiling builds only;
    they cost a memory round trip per phase)."""
    target = Path(out) if out else LIB_PATH
    target.parent.mkdir(parents=True, exist_ok=True)
    tmp = target.with_suffix(".so.tmp")
    flags = [
        f"--offload-arch={ARCH}", "-O3", "-std=c++17", "-fPIC",
        # packed fp32 VALU ops are disabled on purpose (they have produced
        # silent wrong results on this hardware pool)
        "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
        f"-I{INCLUDE}", f"-I{CSRC}",
        *(["-DDSA_PHASE_STAMPS"] if phase_stamps else []),
    ]
    errs = []
    with tempfile.TemporaryDirectory() as d:  # the sources compile side by side
        objs = [Path(d) / (Path(s).stem + ".o") for s in SOURCES]
        procs = [subprocess.Popen([hipcc(), *flags, "-c", str(CSRC / s), "-o", str(o)], stderr=subprocess.PIPE,
                                  text=True) for s, o in zip(SOURCES, objs)]
        for p in procs:
            errs.append(p.communicate()[1])
            if p.returncode != 0:
                raise RuntimeError(f"hipcc failed ({p.returncode}):\n{errs[-1][-4000:]}")
        res = subprocess.run([hipcc(), f"--offload-arch={ARCH}", "-shared", *map(str, objs), "-o", str(tmp)],
                             capture_output=True, text=True)
        if res.returncode != 0:
            raise RuntimeError(f"hipcc failed ({res.returncode}):\n{res.stderr[-4000:]}")
    if verbose:
        print("".join(errs) + res.stderr, file=sys.stderr)
    os.replace(tmp, target)
    return target


if __name__ == "__main__":
    print(build(verbose=True))
