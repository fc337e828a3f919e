"""Builds the host side of one of the library's .hip files against
hip_stub.cpp, a stand-in for the HIP runtime: what an entry point allocates,
copies and launches can then be checked on the CPU, failures included."""
import ctypes as C
import os
import re
import subprocess

from conftest import ROOT

HIPCC = os.path.join(os.environ.get("ROCM_PATH", "/opt/rocm"), "bin", "hipcc")


def build(unit, out_dir):
    """csrc/<unit>.hip and the stand-in as a shared library, loaded."""
    inc = ["-I", os.path.join(ROOT, "include"), "-I", os.path.join(ROOT, "phasecon_amd", "csrc")]
    obj, stub = (os.path.join(out_dir, n) for n in (unit + ".o", "stub.o"))
    subprocess.run([HIPCC, "-O1", "-std=c++17", "-fPIC", "-w", "--offload-arch=gfx950",
                    "--offload-host-only", *inc, "-c",
                    os.path.join(ROOT, "phasecon_amd", "csrc", unit + ".hip"), "-o", obj],
                   check=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(os.path.dirname(os.path.dirname(HIPCC)), "include"), "-c",
                    os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", stub], check=True)
    # the device code, which a host-only object names and does not hold
    names = subprocess.run(["nm", "-u", obj], check=True, capture_output=True, text=True).stdout
    fat = re.findall(r"\b(__hip_fatbin\w*)", names)
    lib = os.path.join(out_dir, unit + "_host.so")
    subprocess.run(["g++", "-shared", "-pthread", "-Wl,-Bsymbolic", "-o", lib, obj, stub,
                    *[f"-Wl,--defsym={f}=0" for f in fat]], check=True)
    L = C.CDLL(lib)
    for f in ("launches", "mallocs", "pins", "live", "live_pins", "live_events"):
        getattr(L, "stub_" + f).restype = C.c_longlong
    L.stub_fail_malloc.argtypes = [C.c_longlong]
    L.stub_log.restype = C.c_char_p
    return L


def launches(L):
    """(kernel, grid x, y, z, threads) of the launches since the last clear."""
    rows = (r.rsplit(" ", 4) for r in L.stub_log().decode().splitlines())
    return [(r[0], *map(int, r[1:])) for r in rows]
