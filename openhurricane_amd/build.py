"""Build libohc.so (host C++17 + HIP kernels for gfx950) in-tree.

Steps:
  1. g++ builds the host-only code generator ohc_codegen (mechanism loader +
     descriptor emitter);
  2. ohc_codegen turns each shipped mechanism into a compile-time descriptor
     header and a registry translation unit is written;
  3. hipcc compiles the kernels and the C-ABI for gfx950 and links
     openhurricane_amd/libohc.so.

Run as ``python -m openhurricane_amd.build`` or through __graft_entry__.build().
"""
from __future__ import annotations

import os
import shutil
import subprocess
import time
import sys
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = PKG / "_build"
GEN = BUILD / "gen"
LIB = PKG / "libohc.so"
ROCM = Path(os.environ.get("ROCM_PATH", "/opt/rocm"))
ARCH = os.environ.get("OHC_OFFLOAD_ARCH", "gfx950")

# Mechanisms that get compile-time specialised lane kernels: name -> files in data/.
SHIPPED = {
    "h2air": ("h2air/mech.che", "h2air/thermo.dat", "h2air/transport.dat"),
}

HOST_SRCS = ["mech.cpp", "codegen.cpp", "synth.cpp"]

# Padded ODE sizes of the generic kernels (must match wave_dispatch.hip).
WAVE_SIZES = [12, 16, 24, 33, 40, 48, 55, 64]

CXXFLAGS = ["-O2", "-std=c++17", "-fPIC", "-Wall", "-Wextra", "-Wno-unused-parameter"]
HIPFLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}",
    # keep the compiler from emitting packed FP32 instructions
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wno-unused-parameter", "-Wno-unused-result",
    # the lane kernels materialise hundreds of FP64 mechanism constants; hoisting
    # them out of the persistent loop keeps them live through the Jacobian and
    # the LU and forces scratch spills, so machine LICM is off (the generic
    # 33-row integrator also runs 8 % slower with it on)
    "-mllvm", "-disable-machine-licm",
]


def _run(cmd, **kw):
    print("+", " ".join(str(c) for c in cmd), flush=True)
    subprocess.run([str(c) for c in cmd], check=True, **kw)


def build(verbose: bool = True) -> Path:
    hipcc = shutil.which("hipcc") or str(ROCM / "bin" / "hipcc")
    gxx = shutil.which("g++") or "g++"
    BUILD.mkdir(exist_ok=True)
    GEN.mkdir(exist_ok=True)
    # 1. code generator
    tool = BUILD / "ohc_codegen"
    _run([gxx, *CXXFLAGS, "-o", tool, *(CSRC / s for s in HOST_SRCS + ["codegen_main.cpp"])])
    # 2. descriptors + registry
    data = PKG / "data"
    entries = []
    for name, (ck, th, tr) in SHIPPED.items():
        out = GEN / f"mech_{name}.h"
        _run([tool, name, data / ck, data / th, data / tr, out])
        entries.append(name)
    reg = GEN / "lane_registry.hip"
    lines = ['// Generated by build.py -- registry of specialised lane kernels.',
             '#include "lane_kernels.hpp"', '#include "quad_lane.hpp"']
    lines += [f'#include "mech_{n}.h"' for n in entries]
    lines += ["", "static const ohcd::LaneEntry kEntries[] = {"]
    lines += [f'    ohcd::LaneLaunch<Mech_{n}>::entry("{n}"),' for n in entries]
    lines += ["};", "",
              'extern "C" const ohcd::LaneEntry *ohc_lane_entries(int *count) {',
              "    *count = (int)(sizeof(kEntries) / sizeof(kEntries[0]));",
              "    return kEntries;", "}"]
    reg.write_text("\n".join(lines) + "\n")
    # 3. objects + link
    objs = []
    for s in HOST_SRCS:
        o = BUILD / (Path(s).stem + ".o")
        _run([gxx, *CXXFLAGS, "-O3", "-c", CSRC / s, "-o", o])
        objs.append(o)
    # The compiled lane kernels sum into accumulators that start at 0.0 and run
    # Horner chains whose lowest coefficient is 0; without signed zeros those
    # adds fold away (only the sign of an exact zero result can change).
    jobs = [(src, BUILD / (src.stem + ".hip.o"), ["-fno-signed-zeros"] if src == reg else [])
            for src in [CSRC / "ohc_api.cpp", reg, CSRC / "wave_dispatch.hip",
                        CSRC / "props_table.hip", CSRC / "source_table.hip",
                        CSRC / "surrogate_api.hip", CSRC / "sched.hip", CSRC / "noalloc.hip"]]
    jobs += [(CSRC / "wave_size.hip", BUILD / f"wave_{n}.hip.o", [f"-DOHC_WAVE_N={n}"])
             for n in WAVE_SIZES]
    procs = []
    width = max(1, min(len(jobs), os.cpu_count() or 4))
    for src, o, extra in jobs:
        cmd = [hipcc, *HIPFLAGS, *extra, f"-I{CSRC}", "-x", "hip", "-c", src, "-o", o]
        print("+", " ".join(str(c) for c in cmd), flush=True)
        while sum(p.poll() is None for p in procs) >= width:
            time.sleep(0.2)
        procs.append(subprocess.Popen([str(c) for c in cmd]))
        objs.append(o)
    bad = [p.args for p in procs if p.wait() != 0]
    if bad:
        raise subprocess.CalledProcessError(1, bad[0])
    tmp = LIB.with_suffix(".so.tmp")
    _run([hipcc, "-shared", f"--offload-arch={ARCH}", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    build()
    print(LIB)
    sys.exit(0)
