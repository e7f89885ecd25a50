"""Builds libseqan_amd.so in-tree with hipcc for gfx950.

    python -m seqan_amd.build            # or: python seqan_amd/build.py

The shared library holds the HIP kernels, the host engine behind the C ABI
(include/seqan_amd.h), the scoring presets and the synthetic workload
generator.  It is built next to this file so that it travels with the tree.
"""
from __future__ import annotations

import json
import concurrent.futures
import os
import shutil
import subprocess
import sys

PKG = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(PKG)
CSRC = os.path.join(PKG, "csrc")
LIB = os.path.join(PKG, "libseqan_amd.so")
ARCH = os.environ.get("SQMI_OFFLOAD_ARCH", "gfx950")

# (source, object name, defines).  score16.hip and band16.hip are built once per
# DNA profile / substitution table and kind, trace16.hip per profile / table; the sources
# compile in parallel, the longest first.
SOURCES = [("score16.hip", f"score16_{t}_{k}", {"SQMI_SCORE_DNA": d, "SQMI_SCORE_KIND": f"kScore{k}",
                                                "SQMI_SCORE_PART": f"score{t}{k}"})
           for d, t in ((0, "Tab"), (1, "Dna")) for k in ("Local", "Right", "Global")]
SOURCES += [("band16.hip", f"band16_{t}_{k}", {"SQMI_BAND_DNA": d, "SQMI_BAND_KIND": f"kBand{k}",
                                              "SQMI_BAND_PART": f"band{t}{k}"})
            for d, t in ((0, "Tab"), (1, "Dna")) for k in ("Local", "Free", "End")]
SOURCES += [("trace16.hip", "trace16_tab", {"SQMI_TRACE_DNA": 0, "SQMI_TRACE_PART": "traceTab"}),
            ("trace16.hip", "trace16_dna", {"SQMI_TRACE_DNA": 1, "SQMI_TRACE_PART": "traceDna"}),
            ("kernels.hip", "kernels", {}), ("lane.hip", "lane", {}),
            ("long16.hip", "long16", {}), ("long.hip", "long", {}), ("banded.hip", "banded", {}), ("scratch.hip", "scratch", {}),
            ("engine.cpp", "engine", {}), ("scoring.cpp", "scoring", {}), ("workload.cpp", "workload", {})]
JOBS = max(1, min(8, os.cpu_count() or 1))


def hipcc():
    for cand in (os.environ.get("HIPCC"), "/opt/rocm/bin/hipcc", shutil.which("hipcc")):
        if cand and os.path.exists(cand):
            return cand
    raise FileNotFoundError("hipcc not found")


SHAPE_TABLE = os.path.join(PKG, "tuning", "shapes.json")
CATEGORIES = ["dna", "dna_local", "table", "table_local"]
NBINS = 16


def shape_table_source(path: str = SHAPE_TABLE) -> str:
    """C++ initializers of the planner's shape table (length bin x count
    class -> groups or rows per lane), from the committed JSON table."""
    with open(path) as f:
        t = json.load(f)
    shapes = [tuple(int(x) for x in s) for s in t["shapes"]]
    classes = [int(c) for c in t["count_classes"]]
    if not shapes or not classes or classes[0] != 0 or sorted(classes) != classes or len(classes) > 4:
        raise ValueError(f"{path}: bad shapes or count_classes")
    rows = []
    for cat in CATEGORIES:
        bins = t["categories"][cat]
        if len(bins) != NBINS or any(len(b) != len(classes) for b in bins):
            raise ValueError(f"{path}: category {cat} needs {NBINS} bins x {len(classes)} classes")
        for b in bins:
            if any(not 0 <= int(x) < len(shapes) for x in b):
                raise ValueError(f"{path}: category {cat}: shape index out of range")
        rows.append("{" + ", ".join("{" + ", ".join(str(int(x)) for x in b + [0] * (4 - len(b))) + "}"
                                    for b in bins) + "}")
    prov = json.dumps(t.get("provenance", {}), sort_keys=True).replace("\\", "\\\\").replace('"', '\\"')
    return "\n".join([
        "// Generated by seqan_amd/build.py from seqan_amd/tuning/shapes.json; do not edit.",
        "constexpr int kTabShapes[][2] = {" + ", ".join(f"{{{g}, {r}}}" for g, r in shapes) + "};",
        f"constexpr int kTabNClasses = {len(classes)};",
        "constexpr int64_t kTabCountClasses[4] = {" + ", ".join(str(c) for c in classes + [0] * (4 - len(classes))) + "};",
        "constexpr uint8_t kTabChoice[4][16][4] = {" + ",\n    ".join(rows) + "};",
        f'constexpr const char *kTabProvenance = "{prov}";',
        ""])


def build(verbose: bool = False) -> str:
    cc = hipcc()
    objdir = os.path.join(PKG, "_build")
    os.makedirs(objdir, exist_ok=True)
    with open(os.path.join(objdir, "shape_table.inc"), "w") as f:
        f.write(shape_table_source())
    common = ["-O3", "-std=c++17", "-fPIC", "-Wall", "-Wno-unused-result",
              f"-I{os.path.join(ROOT, 'include')}", f"-I{CSRC}", f"-I{objdir}"]
    def compile_one(entry):
        src, name, defs = entry
        path = os.path.join(CSRC, src)
        obj = os.path.join(objdir, name + ".o")
        cmd = [cc] + common + [f"-D{k}={v}" for k, v in defs.items()]
        if src.endswith(".hip"):
            # Device code: gfx950 only; packed FP32 instructions disabled.
            cmd += [f"--offload-arch={ARCH}", "-x", "hip",
                    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops"]
        else:
            cmd += ["-x", "c++", "-fopenmp", "-D__HIP_PLATFORM_AMD__", "-I/opt/rocm/include"]
        cmd += ["-c", path, "-o", obj]
        if verbose:
            print(" ".join(cmd), flush=True)
        r = subprocess.run(cmd, capture_output=True, text=True)
        return obj, src, r

    objs = []
    with concurrent.futures.ThreadPoolExecutor(max_workers=JOBS) as pool:
        for obj, src, r in pool.map(compile_one, SOURCES):
            if r.returncode != 0:
                sys.stderr.write(r.stdout + r.stderr)
                raise RuntimeError(f"compiling {src} failed")
            objs.append(obj)
    tmp = LIB + ".tmp"
    link = [cc, "-shared", "-fPIC", "-fopenmp", f"--offload-arch={ARCH}", "-o", tmp] + objs + [
        "-Wl,-rpath,/opt/rocm/lib", "-Wl,-rpath,/opt/rocm/lib/llvm/lib", "-Wl,-rpath,/opt/rocm/llvm/lib"]
    if verbose:
        print(" ".join(link), flush=True)
    r = subprocess.run(link, capture_output=True, text=True)
    if r.returncode != 0:
        sys.stderr.write(r.stdout + r.stderr)
        raise RuntimeError("linking libseqan_amd.so failed")
    os.replace(tmp, LIB)
    return LIB


if __name__ == "__main__":
    print(build(verbose="-v" in sys.argv))
