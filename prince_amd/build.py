"""In-tree build of libprince_hip.so for gfx950 (hipcc, no cmake).

Usage: ``python -m prince_amd.build``.  The shared library lands next to
``prince_amd/_lib.py`` so it travels with the source tree.
"""

from __future__ import annotations

import os
import shutil
import subprocess
import sys
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
SOURCES = [os.path.join(CSRC, f) for f in ("prince_hip.hip", "team_march.hip")]
OUT = os.path.join(HERE, "libprince_hip.so")

HIPCC_FLAGS = [
    "--offload-arch=gfx950",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Xclang",
    "-target-feature",
    "-Xclang",
    "-packed-fp32-ops",
    "-I" + os.path.join(ROOT, "include"),
]

# the march holds its state in 128 registers: constants of exp() and the like
# hoisted out of its step loop would spill (26 registers of scratch per wave)
SOURCE_FLAGS = {"team_march.hip": ["-mllvm", "-disable-machine-licm"]}


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise RuntimeError("hipcc not found (ROCm toolchain required)")


def build(verbose=False):
    """Compile every source (in parallel) and link the shared library."""
    cc = hipcc()
    with tempfile.TemporaryDirectory() as tmpdir:
        objs = [os.path.join(tmpdir, os.path.basename(s) + ".o") for s in SOURCES]
        procs = [subprocess.Popen([cc, *HIPCC_FLAGS,
                                   *SOURCE_FLAGS.get(os.path.basename(s), []), "-c", "-o", o, s], stdout=subprocess.PIPE,
                                  stderr=subprocess.STDOUT, text=True)
                 for s, o in zip(SOURCES, objs)]
        outs = [p.communicate()[0] for p in procs]
        tmp = OUT + ".tmp"
        ok = all(p.returncode == 0 for p in procs)
        if ok:
            res = subprocess.run([cc, "--offload-arch=gfx950", "-shared", "-o", tmp, *objs],
                                 capture_output=True, text=True)
            outs.append(res.stdout + res.stderr)
            ok = res.returncode == 0
        if not ok:
            sys.stderr.write("".join(outs))
            raise RuntimeError("hipcc failed building libprince_hip.so")
        if verbose:
            sys.stdout.write("".join(outs))
        os.replace(tmp, OUT)
    return OUT


if __name__ == "__main__":
    print(build(verbose=True))
