"""The library's host side against hip_stub.cpp, a stand-in for the HIP
runtime: what an entry point allocates, copies and launches can then be
checked on the CPU, failures included."""
import ctypes as C
import functools
import os
import re
import shutil
import subprocess
import tempfile

from conftest import ROOT

ROCM = os.environ.get("ROCM_PATH", "/opt/rocm")
HIPCC = os.path.join(ROCM, "bin", "hipcc")


@functools.lru_cache(None)
def library():
    """Both libraries' sources and the stand-in as one shared library."""
    out = tempfile.mkdtemp(prefix="hip_stub_")
    src, inc = os.path.join(ROOT, "phasecon_amd", "csrc"), os.path.join(ROOT, "include")
    at = lambda n: os.path.join(out, n)  # noqa: E731
    units = ("mbir_hip", "unet_hip", "pcmbir_hip")
    hip = [subprocess.Popen([HIPCC, "-O1", "-std=c++17", "-fPIC", "-w", "--offload-arch=gfx950",
                             "--offload-host-only", "-I", inc, "-c",
                             os.path.join(src, u + ".hip"), "-o", at(u + ".o")]) for u in units]
    for u in ("mbir_engine", "pcmbir_engine"):
        subprocess.run(["gcc", "-O1", "-std=gnu11", "-fPIC", "-w", "-I", inc,
                        "-I", os.path.join(ROCM, "include"), "-c", os.path.join(src, u + ".c"),
                        "-o", at(u + ".o")], check=True)
    subprocess.run(["g++", "-O1", "-std=c++17", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I", os.path.join(ROCM, "include"), "-c",
                    os.path.join(ROOT, "tests", "hip_stub.cpp"), "-o", at("stub.o")], check=True)
    assert [p.wait() for p in hip] == [0] * len(units)
    objs = [at(u + ".o") for u in units + ("mbir_engine", "pcmbir_engine", "stub")]
    # the device code, which a host-only object names and does not hold
    names = subprocess.run(["nm", "-u", *objs], check=True, capture_output=True, text=True).stdout
    fat = set(re.findall(r"\b(__hip_fatbin\w*)", names))
    subprocess.run(["g++", "-shared", "-pthread", "-Wl,-Bsymbolic", "-o", at("host.so"), *objs,
                    "-lm", *[f"-Wl,--defsym={f}=0" for f in fat]], check=True)
    L = C.CDLL(at("host.so"))
    shutil.rmtree(out)
    for f in ("launches", "mallocs", "pins", "live", "live_pins", "live_events"):
        getattr(L, "stub_" + f).restype = C.c_longlong
    L.stub_fail_malloc.argtypes = [C.c_longlong]
    L.stub_log.restype = C.c_char_p
    return L


def use(monkeypatch):
    """Has the package's modules call the stand-in's library; returns it."""
    from phasecon_amd import lib, pcmbir
    L = library()
    for mod in (lib, pcmbir):
        for name, (res, args) in mod._SIGS.items():
            fn = getattr(L, name)
            fn.restype = res
            if args is not None:
                fn.argtypes = args
        monkeypatch.setattr(mod, "_LIB", L)
    L.stub_fail_malloc(-1)
    L.stub_clear_log()
    return L


def launches(L):
    """(kernel, grid x, y, z, threads) of the launches since the last clear."""
    rows = (r.rsplit(" ", 4) for r in L.stub_log().decode().splitlines())
    return [(r[0], *map(int, r[1:])) for r in rows]
