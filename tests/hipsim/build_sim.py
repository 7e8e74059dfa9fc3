"""Build tests/hipsim/libmoshi_sim.so: the SAME engine/kernel sources as the product library, compiled for the
host against the hipsim fiber simulator.  TEST INFRASTRUCTURE ONLY - used by `-m "not gpu"` tests to exercise the
kernel logic (indexing, ring state, masks, packing, reductions) where no GPU exists.  The product never loads it.
"""
from __future__ import annotations

import os
import subprocess
import sys
from pathlib import Path

HERE = Path(__file__).resolve().parent
ROOT = HERE.parent.parent
CSRC = ROOT / "moshi_amd" / "csrc"
LIB = HERE / "libmoshi_sim.so"
TLM_LIB = HERE / "libmoshi_tlm_sim.so"
SOURCES = ["api_common.hip", "mimi_engine.hip", "lm_engine.hip", "batcher.hip", "duplex.hip"]
TLM_SOURCES = ["api_common.hip", "tlm_engine.hip"]


def _cxx() -> str:
    for cand in (os.environ.get("HIPSIM_CXX"), "/opt/rocm/lib/llvm/bin/clang++", "clang++"):
        if cand and (not os.path.isabs(cand) or os.path.exists(cand)):
            return cand
    raise RuntimeError("clang++ not found")


def needs_build(lib: Path = LIB) -> bool:
    if not lib.exists():
        return True
    t = lib.stat().st_mtime
    deps = (list(CSRC.glob("*.h")) + list(CSRC.glob("*.hip")) + list(HERE.glob("*.h")) + list(HERE.glob("*.cpp")) +
            list((ROOT / "include").glob("*.h")))
    return any(p.stat().st_mtime > t for p in deps)


def build_tlm(force: bool = False, verbose: bool = False) -> Path:
    """The token-LM library (libmoshi_tlm.so's sources) on the simulator."""
    return build(force, verbose, TLM_LIB, TLM_SOURCES)


def build(force: bool = False, verbose: bool = False, lib: Path = LIB, sources=None) -> Path:
    """Several test workers may call this at once: the compile runs under a file lock."""
    import fcntl
    with open(HERE / ".build.lock", "w") as lock:
        fcntl.flock(lock, fcntl.LOCK_EX)
        try:
            return _build_locked(force, verbose, lib, SOURCES if sources is None else sources)
        finally:
            fcntl.flock(lock, fcntl.LOCK_UN)


def _build_locked(force: bool, verbose: bool, lib: Path, sources) -> Path:
    if not force and not needs_build(lib):
        return lib
    objs, jobs = [], []
    common = [_cxx(), "-O2", "-g", "-std=c++17", "-fPIC", "-ffp-contract=off", "-pthread", "-Wno-unused-value",
              f"-I{HERE}", f"-I{CSRC}"]
    for name in sources:
        src = CSRC / name
        if not src.exists():
            continue
        obj = HERE / (src.stem + ".sim.o")
        cmd = common + ["-x", "c++", "-c", str(src), "-o", str(obj)]
        if verbose:
            print(" ".join(cmd), flush=True)
        jobs.append((subprocess.Popen(cmd), cmd))
        objs.append(obj)
    obj = HERE / "hipsim.sim.o"
    cmd = common + ["-c", str(HERE / "hipsim.cpp"), "-o", str(obj)]
    jobs.append((subprocess.Popen(cmd), cmd))
    objs.append(obj)
    for p, cmd in jobs:
        if p.wait() != 0:
            raise RuntimeError("sim build failed: " + " ".join(cmd))
    cmd = [_cxx(), "-shared", "-fPIC", "-pthread", "-o", str(lib)] + [str(o) for o in objs]
    subprocess.check_call(cmd)
    return lib


def build_asan(out_dir: Path) -> Path:
    """An AddressSanitizer build of the simulator library (every hipMalloc is its own heap block there, so a kernel reading or
    writing past a buffer is reported with the kernel's source line).  Run the simulator suites on it with

        python tests/hipsim/build_sim.py --asan /tmp/asan
        LD_PRELOAD=$(dirname $(dirname /opt/rocm/lib/llvm/bin))/lib/clang/*/lib/linux/libclang_rt.asan-x86_64.so \
        ASAN_OPTIONS=detect_leaks=0:detect_stack_use_after_return=0 MMI_SIM_LIB=/tmp/asan/libmoshi_sim_asan.so \
        python -m pytest tests/test_mimi_sim.py tests/test_lm_sim.py tests/test_batcher_sim.py tests/test_duplex_sim.py -m "not gpu"

    (no report; the one failure is test_io_threads_push_and_pop..., whose 60 s deadline the 5x slower
    instrumented build misses)."""
    out_dir.mkdir(parents=True, exist_ok=True)
    flags = [_cxx(), "-O1", "-g", "-std=c++17", "-fPIC", "-ffp-contract=off", "-pthread", "-Wno-unused-value", "-Wno-psabi",
             "-fsanitize=address", "-fno-omit-frame-pointer", "-DHIPSIM_UCONTEXT", f"-I{HERE}", f"-I{CSRC}"]
    jobs, objs = [], []
    for name in SOURCES:
        obj = out_dir / (Path(name).stem + ".asan.o")
        jobs.append(subprocess.Popen(flags + ["-x", "c++", "-c", str(CSRC / name), "-o", str(obj)]))
        objs.append(obj)
    obj = out_dir / "hipsim.asan.o"
    jobs.append(subprocess.Popen(flags + ["-c", str(HERE / "hipsim.cpp"), "-o", str(obj)]))
    objs.append(obj)
    if any(p.wait() != 0 for p in jobs):
        raise RuntimeError("asan sim build failed")
    lib = out_dir / "libmoshi_sim_asan.so"
    subprocess.check_call([_cxx(), "-shared", "-fPIC", "-pthread", "-fsanitize=address", "-shared-libasan", "-o", str(lib)] + [str(o) for o in objs])
    return lib


def build_ubsan(out_dir: Path) -> Path:
    """An UndefinedBehaviorSanitizer build of the simulator library (signed overflow, shifts out of range, misaligned or null
    accesses, out-of-range float -> int conversions, array indexing past a declared bound in the kernel and engine sources):

        python tests/hipsim/build_sim.py --ubsan /tmp/ubsan
        LD_PRELOAD=$(dirname $(dirname /opt/rocm/lib/llvm/bin))/lib/clang/*/lib/linux/libclang_rt.ubsan_standalone-x86_64.so \
        UBSAN_OPTIONS=print_stacktrace=1:log_path=/tmp/ubsan/report MMI_SIM_LIB=/tmp/ubsan/libmoshi_sim_ubsan.so \
        python -m pytest tests/test_mimi_sim.py tests/test_lm_sim.py tests/test_batcher_sim.py tests/test_duplex_sim.py -m "not gpu"

    Reports are recoverable (the suite runs to its end) and land in /tmp/ubsan/report.<pid>."""
    out_dir.mkdir(parents=True, exist_ok=True)
    flags = [_cxx(), "-O1", "-g", "-std=c++17", "-fPIC", "-ffp-contract=off", "-pthread", "-Wno-unused-value", "-Wno-psabi",
             "-fsanitize=undefined,float-cast-overflow", "-fno-omit-frame-pointer", "-DHIPSIM_UCONTEXT", f"-I{HERE}", f"-I{CSRC}"]
    jobs, objs = [], []
    for name in SOURCES:
        obj = out_dir / (Path(name).stem + ".ubsan.o")
        jobs.append(subprocess.Popen(flags + ["-x", "c++", "-c", str(CSRC / name), "-o", str(obj)]))
        objs.append(obj)
    obj = out_dir / "hipsim.ubsan.o"
    jobs.append(subprocess.Popen(flags + ["-c", str(HERE / "hipsim.cpp"), "-o", str(obj)]))
    objs.append(obj)
    if any(p.wait() != 0 for p in jobs):
        raise RuntimeError("ubsan sim build failed")
    lib = out_dir / "libmoshi_sim_ubsan.so"
    subprocess.check_call([_cxx(), "-shared", "-fPIC", "-pthread", "-fsanitize=undefined,float-cast-overflow", "-shared-libsan",
                           "-o", str(lib)] + [str(o) for o in objs])
    return lib


if __name__ == "__main__":
    if "--asan" in sys.argv:
        print(build_asan(Path(sys.argv[sys.argv.index("--asan") + 1])))
        sys.exit(0)
    if "--ubsan" in sys.argv:
        print(build_ubsan(Path(sys.argv[sys.argv.index("--ubsan") + 1])))
        sys.exit(0)
    build(force="--force" in sys.argv, verbose=True)
    print(LIB)
