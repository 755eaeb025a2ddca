"""Builds the native library in-tree: bigstickpublick_amd/libbigstick_amd.so
(hipcc, gfx950) and the Fortran iso_c_binding module when amdflang exists."""
import os
import shutil
import subprocess
import tempfile

HERE = os.path.dirname(os.path.abspath(__file__))
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libbigstick_amd.so")
HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")

HIP_FLAGS = [
    "--offload-arch=gfx950", "-O3", "-std=c++17", "-fPIC", "-shared",
    # packed FP32 instructions stay off (see the engine's build notes)
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-ffp-contract=off", "-Wall", "-Wno-unused-result",
]


SOURCES = ("bs_engine.hip", "bs_like.hip", "bs_short.hip", "bs_tables.cpp")


def build_native(verbose=False):
    """Compiles every source (side by side) and links the library."""
    bdir = os.path.join(CSRC, "_build")
    os.makedirs(bdir, exist_ok=True)
    inc = ["-I", os.path.join(os.path.dirname(HERE), "include")]
    jobs = []
    for src in SOURCES:
        obj = os.path.join(bdir, src + ".o")
        cmd = [HIPCC] + [f for f in HIP_FLAGS if f != "-shared"] + inc + ["-c", os.path.join(CSRC, src), "-o", obj]
        log = tempfile.TemporaryFile(mode="w+")  # (a full pipe would stop the compiler)
        jobs.append((src, obj, log, subprocess.Popen(cmd, stdout=log, stderr=subprocess.STDOUT)))
    failed = []
    for src, obj, log, p in jobs:
        p.wait()
        log.seek(0)
        out = log.read()
        log.close()
        if p.returncode != 0:
            failed.append("%s:\n%s" % (src, out))
        elif verbose:
            print(out)
    if failed:
        raise RuntimeError("hipcc failed:\n" + "\n".join(failed))
    tmp = LIB + ".tmp"
    r = subprocess.run([HIPCC, "--offload-arch=gfx950", "-shared", "-o", tmp] + [j[1] for j in jobs] +
                       ["-lrocsolver", "-lrocblas"], capture_output=True, text=True)
    if r.returncode != 0:
        raise RuntimeError("hipcc failed:\n" + r.stdout + r.stderr)
    os.replace(tmp, LIB)
    return LIB


FORTRAN = os.path.join(HERE, "fortran")
FDRIVER = os.path.join(FORTRAN, "bs_driver")


def build_fortran():
    """The iso_c_binding module and the bs_driver Fortran host (amdflang);
    skipped when no Fortran compiler is installed."""
    fc = os.environ.get("FC_AMD", "/opt/rocm/bin/amdflang")
    if not os.path.exists(fc):
        return None
    bdir = os.path.join(FORTRAN, "_build")
    os.makedirs(bdir, exist_ok=True)
    steps = [
        [fc, "-O2", "-c", os.path.join(FORTRAN, "bigstick_amd.f90"), "-o",
         os.path.join(bdir, "bigstick_amd.o"), "-module-dir", bdir],
        [fc, "-O2", "-I", bdir, os.path.join(FORTRAN, "bs_driver.f90"),
         os.path.join(bdir, "bigstick_amd.o"), "-L", HERE, "-lbigstick_amd",
         "-Wl,-rpath,$ORIGIN/..", "-L/opt/rocm/lib", "-lamdhip64", "-o", FDRIVER + ".tmp"],
    ]
    for cmd in steps:
        r = subprocess.run(cmd, capture_output=True, text=True)
        if r.returncode != 0:
            raise RuntimeError("amdflang failed:\n" + r.stdout + r.stderr)
    os.replace(FDRIVER + ".tmp", FDRIVER)
    return FDRIVER


if __name__ == "__main__":
    print(build_native(verbose=True))
    print(build_fortran())
