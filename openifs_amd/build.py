"""Build the native parts in-tree.

    python -m openifs_amd.build          # libcloudsc_hip.so (gfx950) + the CPU oracle

libcloudsc_hip.so is compiled with hipcc for gfx950 only; the CPU oracle
(test infrastructure) with oracle/Makefile.  Outputs stay in the source tree
(openifs_amd/libcloudsc_hip.so, oracle/liboracle_cloudsc.so) so that they
travel with the repository snapshot.
"""
import os
import subprocess
import sys
from concurrent.futures import ThreadPoolExecutor

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(HERE, "csrc")
LIB = os.path.join(HERE, "libcloudsc_hip.so")
OBJDIR = os.path.join(HERE, "_build")

HIPCC = os.environ.get("HIPCC", "/opt/rocm/bin/hipcc")
ARCH = "gfx950"
HIP_FLAGS = [
    f"--offload-arch={ARCH}",
    "-O3",
    "-std=c++17",
    "-fPIC",
    # No FMA contraction: CLOUDSC compares cancellation residues against ZEPSEC = 1e-14 and
    # tests supersaturation against a limit; fused products change which side of those
    # thresholds FP32 results fall on in almost every column, while unfused arithmetic keeps
    # the FP32 kernel as close to FP64 as the FP32 CPU oracle is.
    "-ffp-contract=off",
    # FP32 exp/pow on v_exp_f32/v_log_f32 (FP64 keeps accurate functions: the library's, in the column sweep its own)
    "-DCLOUDSC_FAST_TRANSCENDENTALS",
    # packed FP32 (v_pk_*_f32) is disabled for all device code
    "-Xclang", "-target-feature", "-Xclang", "-packed-fp32-ops",
    "-I", os.path.join(ROOT, "include"),
]
SOURCES = ["cloudsc_kernel.hip", "cloudsc_capi.hip", "synth.hip", "cloudsc_params.cpp", "mlp.hip", "surrogate.hip",
           "satadj.hip", "field.hip", "supersat.hip", "cloudsc2.hip"]


def _run(cmd, cwd=None):
    r = subprocess.run(cmd, cwd=cwd, stdout=subprocess.PIPE, stderr=subprocess.STDOUT, text=True)
    if r.returncode != 0:
        raise RuntimeError(f"command failed ({r.returncode}): {' '.join(cmd)}\n{r.stdout}")
    return r.stdout


def build_hip(verbose=False):
    os.makedirs(OBJDIR, exist_ok=True)

    def compile_one(src):
        obj = os.path.join(OBJDIR, os.path.splitext(src)[0] + ".o")
        cmd = [HIPCC, *HIP_FLAGS, "-x", "hip", "-c", os.path.join(CSRC, src), "-o", obj]
        out = _run(cmd)
        if verbose and out.strip():
            print(out)
        return obj

    with ThreadPoolExecutor(max_workers=len(SOURCES)) as ex:
        objs = list(ex.map(compile_one, SOURCES))
    tmp = LIB + ".tmp"
    _run([HIPCC, f"--offload-arch={ARCH}", "-shared", "-fPIC", "-o", tmp, *objs])
    os.replace(tmp, LIB)
    return LIB


def build_oracle():
    _run(["make", "-s", "-C", os.path.join(ROOT, "oracle")])
    return os.path.join(ROOT, "oracle", "liboracle_cloudsc.so")


DEVICE_CHECK_SRC = os.path.join(ROOT, "tests", "hip", "device_check.hip")
DEVICE_CHECK = os.path.join(ROOT, "tests", "hip", "libdevice_check.so")


def build_device_check():
    """Device functions of the column kernels as a library of their own, for the tests."""
    _run([HIPCC, *HIP_FLAGS, "-shared", "-o", DEVICE_CHECK, DEVICE_CHECK_SRC])
    return DEVICE_CHECK


FLANG = os.environ.get("FLANG", "/opt/rocm/lib/llvm/bin/flang")
FORTRAN_MOD = os.path.join(HERE, "fortran", "cloudsc_hip_mod.F90")
FORTRAN_DRIVER_SRC = os.path.join(ROOT, "tests", "fortran", "cloudsc_fortran_driver.F90")
FORTRAN_DRIVER = os.path.join(ROOT, "tests", "fortran", "cloudsc_fortran_driver")


def build_fortran():
    """The ISO_C_BINDING module and the Fortran host driver used by the tests (needs flang)."""
    if not os.path.exists(FLANG):
        return None
    fdir = os.path.join(OBJDIR, "fortran")
    os.makedirs(fdir, exist_ok=True)
    mod_o = os.path.join(fdir, "cloudsc_hip_mod.o")
    drv_o = os.path.join(fdir, "cloudsc_fortran_driver.o")
    _run([FLANG, "-O1", "-c", FORTRAN_MOD, "-o", mod_o, "-module-dir", fdir])
    _run([FLANG, "-O1", "-c", FORTRAN_DRIVER_SRC, "-o", drv_o, "-module-dir", fdir, "-I", fdir])
    _run([FLANG, "-o", FORTRAN_DRIVER, drv_o, mod_o, "-L", HERE, "-lcloudsc_hip",
          "-Wl,-rpath,$ORIGIN/../../openifs_amd"])
    return FORTRAN_DRIVER


def build_all(verbose=False):
    lib = build_hip(verbose)
    orc = build_oracle()
    build_device_check()
    build_fortran()
    return lib, orc


if __name__ == "__main__":
    print(build_all(verbose="-v" in sys.argv))
