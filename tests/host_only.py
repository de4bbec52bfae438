"""The library's host code (fgl_host.cpp) over a HIP runtime in host memory
(fake_hip.cpp): tests of what it asks of the runtime, without a GPU."""
import functools
import os
import re
import subprocess
import sys
import tempfile

import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)
CSRC = os.path.join(ROOT, "fauxgl_amd", "csrc")
_dir = None


@functools.lru_cache(None)
def library():
    """Compiles both and links them; the launch entry points of the device
    code that neither defines become functions returning 0."""
    global _dir
    from fauxgl_amd import build as B
    try:
        cc = B.hipcc()
    except RuntimeError:
        pytest.skip("hipcc not found")
    _dir = tempfile.TemporaryDirectory(prefix="fgl_host_only_")
    objs = []
    for src in (os.path.join(CSRC, "fgl_host.cpp"), os.path.join(HERE, "fake_hip.cpp")):
        obj = os.path.join(_dir.name, os.path.basename(src) + ".o")
        subprocess.run([cc, "--offload-arch=gfx950", "-O1", "-std=c++17", "-fPIC", "-ffp-contract=off", "-I", CSRC,
                        "-c", src, "-o", obj], check=True)
        objs.append(obj)
    names = {}
    for obj in objs:
        for ln in subprocess.run(["nm", obj], capture_output=True, text=True, check=True).stdout.splitlines():
            *_, kind, name = ln.split()
            if re.match(r"_ZN3fgl\d", name):
                names[name] = names.get(name, False) or kind != "U"
    stubs = os.path.join(_dir.name, "stubs.c")
    with open(stubs, "w") as f:
        f.writelines(f"long {n}(void) {{ return 0; }}\n" for n, defined in sorted(names.items()) if not defined)
    lib = os.path.join(_dir.name, "libfgl_host_only.so")
    subprocess.run(["gcc", "-c", "-fPIC", stubs, "-o", stubs + ".o"], check=True)
    subprocess.run(["g++", "-shared", "-Wl,-Bsymbolic", "-o", lib, *objs, stubs + ".o", "-lpthread"], check=True)
    return lib


def run(code, **env):
    """Runs a Python program whose fauxgl_amd is over that library; `fake` is
    the library itself, for the fake runtime's own entry points."""
    pre = ("import ctypes, sys\n"
           f"sys.path[:0] = [{ROOT!r}, {HERE!r}]\n"
           "import numpy as np\n"
           "from fauxgl_amd import _native as N, api as A, meshes as M\n"
           "fake = N.load()\n"
           "for n in ('fake_live', 'fake_peak'): getattr(fake, n).restype = ctypes.c_size_t\n"
           "fake.fake_limit.argtypes = [ctypes.c_size_t]\n")
    res = subprocess.run([sys.executable, "-c", pre + code], capture_output=True, text=True, timeout=120,
                         env={**os.environ, "FAUXGL_AMD_LIB": library(), **env})
    assert res.returncode == 0, res.stdout + res.stderr
    return res.stdout
