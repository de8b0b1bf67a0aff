"""Build the gfx950 HIP library `libflash_spacetime.so` and the host extension
`_fst_host` (its file carries Python's ABI tag) in the package directory.

Every kernel instance family is its own translation unit so hipcc runs them
in parallel; the objects are linked into one shared library whose C ABI is
declared in include/flash_spacetime.h. Usage: python -m flash_spacetime_amd.build
"""

from __future__ import annotations

import json
import os
import re
import shutil
import subprocess
import sys
import sysconfig
from concurrent.futures import ThreadPoolExecutor
from pathlib import Path

PKG = Path(__file__).resolve().parent
CSRC = PKG / "csrc"
BUILD = CSRC / "_build"
HEADER = PKG.parent / "include" / "flash_spacetime.h"
LIB = PKG / "libflash_spacetime.so"
HOST_LIB = PKG / f"_fst_host{sysconfig.get_config_var('EXT_SUFFIX')}"

ARCH = os.environ.get("FST_OFFLOAD_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")
FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    "-Wall",
    "-Wno-unused-function",
    # Packed fp32 VALU forms are kept out of the device code.
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
]

DTYPES = {"bf16": "bf16", "f32": "float"}
HEAD_DIMS = (16, 32, 48, 64)


# The bf16 tile rows kernel is built in a unit of its own with the machine
# scheduler's max-ilp strategy (cfg2's rows kernel 0.891 -> 0.873 ms); the
# strategy slowed the cols kernel by up to a third at other shapes and the
# float32 forward by 11 %, so every other unit keeps the default.
ROWS_SCHED = ["-mllvm", "--amdgpu-sched-strategy=max-ilp"]


def source_hash() -> str:
    """First 12 hex digits of the SHA-256 of every source and the C header: the
    build id fst_version reports (the tuner's plan cache keys on it, and the
    host extension is used only with the library of its own build)."""
    import hashlib

    h = hashlib.sha256()
    for p in [p for ext in ("h", "hip", "cpp") for p in sorted(CSRC.glob(f"*.{ext}"))] + [HEADER]:
        h.update(p.name.encode())
        h.update(p.read_bytes())
    return h.hexdigest()[:12]


def _units():
    units = [("capi", CSRC / "fst_capi.hip", [f'-DFST_BUILD_ID="{source_hash()}"'])]
    for tag, ctype in DTYPES.items():
        for d in HEAD_DIMS:
            name = f"{tag}_{d}"
            defs = [f"-DFST_T={ctype}", f"-DFST_D={d}", f"-DFST_NAME={name}"]
            units.append((f"fwd_{name}", CSRC / "fst_fwd_inst.hip", defs))
            if tag == "bf16":
                units.append((f"bwdr_{name}", CSRC / "fst_bwd_inst.hip", defs + ["-DFST_BWD_PART=1"] + ROWS_SCHED))
                units.append((f"bwd_{name}", CSRC / "fst_bwd_inst.hip", defs + ["-DFST_BWD_PART=2"]))
            else:
                units.append((f"bwd_{name}", CSRC / "fst_bwd_inst.hip", defs))
    # The slowest units first, so that none is left running alone at the end.
    units.sort(key=lambda u: not u[0].startswith("bwd_f32"))
    return [u for u in units if u[1].exists()]


def _build_host():
    """Compile csrc/fst_host.cpp, the operators' host path (a Python extension
    against torch's C++ API; no device code). It records the build id and the
    torch it was compiled for, which _lib.host compares."""
    import torch
    from torch.utils import cpp_extension

    tmp = HOST_LIB.with_suffix(".so.tmp")
    cmd = [os.environ.get("CXX", "g++"), "-O2", "-std=c++17", "-shared", "-fPIC", "-Wall",
           "-DTORCH_EXTENSION_NAME=_fst_host", f'-DFST_BUILD_ID="{source_hash()}"',
           f'-DFST_TORCH_VERSION="{torch.__version__}"', f"-D_GLIBCXX_USE_CXX11_ABI={int(torch.compiled_with_cxx11_abi())}"]
    for inc in (*cpp_extension.include_paths(), sysconfig.get_paths()["include"]):
        cmd += ["-isystem", str(inc)]
    cmd += [str(CSRC / "fst_host.cpp"), "-o", str(tmp)]
    cmd += [f"-L{p}" for p in cpp_extension.library_paths()] + ["-lc10", "-ltorch_cpu", "-ltorch", "-ltorch_python"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("host extension failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, HOST_LIB)
    (PKG / "_fst_host.so").unlink(missing_ok=True)  # the untagged file of earlier builds


RESOURCES = BUILD / "kernel_resources.json"
_REMARK = re.compile(r"remark:\s+(Function Name|VGPRs|AGPRs|ScratchSize \[bytes/lane\]|Occupancy \[waves/SIMD\]"
                     r"|LDS Size \[bytes/block\]): (\S+)")
_KEYS = {"VGPRs": "vgpr", "AGPRs": "agpr", "ScratchSize [bytes/lane]": "scratch_bytes",
         "Occupancy [waves/SIMD]": "waves_per_simd", "LDS Size [bytes/block]": "static_lds_bytes"}


def _resources(text):
    """Per-kernel register, scratch and occupancy figures from the compiler's
    kernel-resource-usage remarks of one unit (the code object's own counts)."""
    out, cur = {}, None
    for line in text.splitlines():
        m = _REMARK.search(line)
        if not m:
            continue
        key, val = m.group(1), m.group(2)
        if key == "Function Name":
            cur = out.setdefault(val, {})
        elif cur is not None:
            cur[_KEYS[key]] = int(val)
    return out


def _compile(unit):
    name, src, defs = unit
    obj = BUILD / f"{name}.o"
    cmd = [HIPCC, *FLAGS, *defs, "-c", str(src), "-o", str(obj), "-Rpass-analysis=kernel-resource-usage"]
    res = subprocess.run(cmd, capture_output=True, text=True)
    text = res.stdout + res.stderr
    out = "\n".join(
        line for line in text.splitlines()
        if "packed-fp32-ops" not in line and "-Rpass-analysis=kernel-resource-usage" not in line
    )
    return name, obj, res.returncode, out, _resources(text)


def build(jobs: int | None = None, verbose: bool = False) -> Path:
    """Compile every unit (always) and link the shared library."""
    BUILD.mkdir(parents=True, exist_ok=True)
    units = _units()
    jobs = jobs or min(len(units), max(1, min(16, os.cpu_count() or 1)))
    with ThreadPoolExecutor(max_workers=jobs) as pool:
        host = pool.submit(_build_host)
        results = list(pool.map(_compile, units))
        host.result()
    failed = [r for r in results if r[2] != 0]
    for name, _, rc, out, _ in results:
        if out.strip() and (verbose or rc != 0):
            print(f"--- {name} ---\n{out}", file=sys.stderr)
    if failed:
        raise RuntimeError("hipcc failed for: " + ", ".join(r[0] for r in failed))
    resources = {}
    for r in results:
        resources.update(r[4])
    RESOURCES.write_text(json.dumps(resources, indent=0, sort_keys=True))
    tmp = LIB.with_suffix(".so.tmp")
    cmd = [HIPCC, f"--offload-arch={ARCH}", "-shared", "-o", str(tmp), *(str(r[1]) for r in results)]
    res = subprocess.run(cmd, capture_output=True, text=True)
    if res.returncode != 0:
        raise RuntimeError("link failed:\n" + res.stdout + res.stderr)
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
