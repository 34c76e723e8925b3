"""Build the HIP library in-tree: gpuintegration_amd/libpagani.so (gfx950).

Also builds the test helper library tests/cxx/libreftests.so (the
reference's test integrands through the C++ header API) and the C interop
test program.  Every call recompiles.  Objects go to gpuintegration_amd/_build.
"""
import concurrent.futures
import os
import shutil
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
INCLUDE = os.path.join(ROOT, "include")
BUILD = os.path.join(HERE, "_build")
LIB = os.path.join(HERE, "libpagani.so")
TESTS_CXX = os.path.join(ROOT, "tests", "cxx")
REFTESTS_LIB = os.path.join(TESTS_CXX, "libreftests.so")
C_INTEROP_EXE = os.path.join(TESTS_CXX, "test_integration_from_c")

ARCH = os.environ.get("PAGANI_ARCH", "gfx950")
HIPCC = os.environ.get("HIPCC", shutil.which("hipcc") or "/opt/rocm/bin/hipcc")

# Packed FP32 VALU forms are disabled for all device code.
HIP_FLAGS = [
    "-O3", "-std=c++17", "-fPIC", f"--offload-arch={ARCH}", "-I" + INCLUDE, "-I" + CSRC,
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-Wall", "-Wno-unused-command-line-argument", "-Wno-unknown-warning-option",
]

# source -> extra flags
HIP_SOURCES = {
    "phases.hip": ["-ffp-contract=off"],
    "driver.hip": [],
    "genz_eval.hip": [],
    "interop.hip": [],
    "batch.hip": [],
    "checkpoint.hip": [],
    "mcubes.hip": [],
    "noalloc.hip": [],
    "segments.hip": [],
    "small_loop.hip": [],
}
# sources compiled in several parts (one object each, -DPAGANI_PART=k), side
# by side: their kernel instantiations take minutes in one
PARTS = {"genz_eval.hip": 6, "segments.hip": 3, "small_loop.hip": 4}
CXX_SOURCES = {"rule.cpp": ["-O2", "-ffp-contract=off"],
               "mcubes_grid.cpp": ["-O2", "-ffp-contract=off"]}


def _run(cmd):
    p = subprocess.run(cmd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    out = "\n".join(l for l in p.stdout.splitlines()
                    if "packed-fp32-ops" not in l and "is not a recognized feature" not in l)
    if p.returncode != 0:
        raise RuntimeError(f"build step failed: {' '.join(cmd)}\n{out}")
    return out


TUNING_JSON = os.path.join(HERE, "tuning", "eval_slices.json")
FAMILY_CODES = {"oscillatory": 1, "product_peak": 2, "corner_peak": 3, "gaussian": 4, "c0": 5,
                "discontinuous": 6}
MAX_DIM = 16
SLICE_BUCKETS = 32


def generate_tuning_table():
    """Write the autotuner's measurements (tuning/eval_slices.json, from
    gpuintegration_amd/tune.py) as the C table driver.hip compiles in:
    kTunedSlices[family][ndim][precision][size class], 0 where the rule of
    choose_slices_n decides."""
    import json
    table = {}
    if os.path.exists(TUNING_JSON):
        with open(TUNING_JSON) as f:
            data = json.load(f)
        for row in data.get("tables", []):
            fam = FAMILY_CODES[row["family"]]
            d = int(row["ndim"])
            p = 1 if int(row["precision"]) == 32 else 0
            vals = [0] * SLICE_BUCKETS
            for b, s in row["slices"].items():
                vals[int(b)] = int(s)
            # lists of less than a batch: the smallest measured class's entry
            # for the integrands evaluated by pair or group sums; the others'
            # errors are rounding noise that another wave count would move
            if p == 0 and row["family"] != "oscillatory":
                first = min(int(b) for b in row["slices"])
                vals[:first] = [vals[first]] * first
            table[(fam, d, p)] = vals
    lines = ["// generated by gpuintegration_amd/build.py from tuning/eval_slices.json",
             "static const std::uint8_t kTunedSlices[7][%d][2][%d] = {" % (MAX_DIM + 1,
                                                                          SLICE_BUCKETS)]
    for fam in range(7):
        lines.append(" {")
        for d in range(MAX_DIM + 1):
            rows = []
            for p in range(2):
                vals = table.get((fam, d, p), [0] * SLICE_BUCKETS)
                rows.append("{" + ",".join(str(v) for v in vals) + "}")
            lines.append("  {" + ", ".join(rows) + "},")
        lines.append(" },")
    lines.append("};")
    os.makedirs(BUILD, exist_ok=True)
    path = os.path.join(BUILD, "tuned_slices.inc")
    text = "\n".join(lines) + "\n"
    if not os.path.exists(path) or open(path).read() != text:
        with open(path, "w") as f:
            f.write(text)
    return path


def _compile_hip(src, extra, part=None):
    name = os.path.splitext(src)[0] + ("" if part is None else f".{part}")
    obj = os.path.join(BUILD, name + ".o")
    if part is not None:
        extra = [*extra, f"-DPAGANI_PART={part}"]
    _run([HIPCC, *HIP_FLAGS, "-I" + BUILD, *extra, "-c", os.path.join(CSRC, src), "-o", obj])
    return obj


def _hip_jobs():
    """(source, flags, part) of every object, the sources in parts first: they take longest."""
    parts = [(s, HIP_SOURCES[s], k) for s, n in PARTS.items() for k in range(n)]
    return parts + [(s, f, None) for s, f in HIP_SOURCES.items() if s not in PARTS]


def _compile_cxx(src, extra):
    obj = os.path.join(BUILD, os.path.splitext(src)[0] + ".o")
    _run(["g++", "-std=c++17", "-fPIC", "-Wall", "-I" + INCLUDE, "-I" + CSRC, *extra, "-c",
          os.path.join(CSRC, src), "-o", obj])
    return obj


def build_library(jobs=8):
    os.makedirs(BUILD, exist_ok=True)
    generate_tuning_table()
    with concurrent.futures.ThreadPoolExecutor(max_workers=jobs) as ex:
        futs = [ex.submit(_compile_hip, *job) for job in _hip_jobs()]
        futs += [ex.submit(_compile_cxx, s, f) for s, f in CXX_SOURCES.items()]
        objs = [f.result() for f in futs]
    tmp = LIB + ".tmp"
    _run([HIPCC, "-shared", "-fPIC", f"--offload-arch={ARCH}", *objs, "-o", tmp])
    os.replace(tmp, LIB)
    return LIB


HEADER_BENCH_LIB = os.path.join(HERE, "libpagani_header_bench.so")


def build_header_bench():
    """The benchmark's generic leg: a plain functor through the C++ header,
    compiled as a user translation unit against libpagani.so."""
    src = os.path.join(CSRC, "header_bench.hip")
    tmp = HEADER_BENCH_LIB + ".tmp"
    _run([HIPCC, *HIP_FLAGS, "-shared", src, "-L" + HERE, "-lpagani",
          "-Wl,-rpath,$ORIGIN", "-o", tmp])
    os.replace(tmp, HEADER_BENCH_LIB)
    return HEADER_BENCH_LIB


def build_tests():
    src = os.path.join(TESTS_CXX, "reftests.hip")
    if not os.path.exists(src):
        return None
    tmp = REFTESTS_LIB + ".tmp"
    _run([HIPCC, *HIP_FLAGS, "-shared", src, "-L" + HERE, "-lpagani",
          "-Wl,-rpath,$ORIGIN/../../gpuintegration_amd", "-o", tmp])
    os.replace(tmp, REFTESTS_LIB)
    csrc = os.path.join(TESTS_CXX, "test_integration_from_c.c")
    if os.path.exists(csrc):
        _run(["gcc", "-O2", "-Wall", "-I" + INCLUDE, csrc, "-L" + HERE, "-lpagani",
              "-Wl,-rpath," + "$ORIGIN/../../gpuintegration_amd", "-o", C_INTEROP_EXE, "-lm"])
    return REFTESTS_LIB


def build_all():
    build_library()
    with concurrent.futures.ThreadPoolExecutor(max_workers=2) as ex:
        futs = [ex.submit(build_header_bench), ex.submit(build_tests)]
        for f in futs:
            f.result()


if __name__ == "__main__":
    build_all()
    print(LIB)
    sys.exit(0)
