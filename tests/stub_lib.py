"""The library's host code on a stand-in for the HIP runtime (tests/hip_stub): what it launches,
allocates and copies can be followed, and made to fail, without a device."""
import ctypes as C
import os
import subprocess

import pytest

from trans_amd import build, capi

HERE = os.path.dirname(os.path.abspath(__file__))
OUT = os.path.join(HERE, "_build")
LIB = os.path.join(OUT, "libtrans_stub.so")
STUB = os.path.join(HERE, "hip_stub", "hip_stub.hip")


def _stale():
    src = [STUB, os.path.join(HERE, "..", "include", "trans_hip.h")]
    csrc = os.path.dirname(build.SRC)
    src += [os.path.join(csrc, f) for f in os.listdir(csrc)]
    return not os.path.exists(LIB) or any(os.path.getmtime(s) > os.path.getmtime(LIB) for s in src)


def _compile():
    os.makedirs(OUT, exist_ok=True)
    tag = os.path.join(OUT, f"{os.getpid()}")
    host = ["-O1", "-std=c++17", "-fPIC", "-w", "-ffp-contract=off"]
    objs = [tag + "_lib.o", tag + "_stub.o"]
    for src, obj in zip((build.SRC, STUB), objs):
        subprocess.run([build.HIPCC, "--offload-host-only"] + host + ["-c", src, "-o", obj], check=True)
    # the name of the embedded device code, which is left out
    nm = subprocess.run(["nm", "-u", objs[0]], check=True, capture_output=True, text=True).stdout
    fat = [w for w in nm.split() if w.startswith("__hip_fatbin")]
    subprocess.run(["g++", "-shared", "-o", tag + ".so"] + objs + ["-pthread", "-Wl,-Bsymbolic", "-Wl,-z,defs"] +
                   [f"-Wl,--defsym,{f}=0" for f in fat], check=True)
    os.replace(tag + ".so", LIB)
    for obj in objs:
        os.remove(obj)


@pytest.fixture
def stub(monkeypatch):
    """The library on the stand-in runtime, in place of the one the package loads."""
    if _stale():
        _compile()
    monkeypatch.setattr(capi, "_lib", None)
    lib = capi.load_library(LIB)  # (the package's own library comes back after the test)
    lib.stub_log.restype = C.c_char_p
    lib.stub_fail_new.argtypes = [C.c_long]
    lib.stub_new_left.restype = C.c_long
    lib.stub_mapped.restype = C.c_size_t
    lib.stub_reset()
    yield lib
    lib.stub_reset()


def events(lib):
    """(what, name, stream or event) of everything recorded since the reset."""
    return [tuple(line.split()) for line in lib.stub_log().decode().splitlines()]
