"""Runs libquickfock.so on the CPU over mock_hip.cpp: launches are recorded and
kernels do nothing.  ``run(code)`` executes Python source in a child process
that holds no other HIP runtime; there ``start()`` returns the mock and
``launches(mock)`` what it recorded."""
import collections
import ctypes
import os
import re
import subprocess
import sys

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

Launch = collections.namedtuple("Launch", "name grid slots deps before")


def build(folder):
    so = os.path.join(str(folder), "mock_hip.so")
    subprocess.run(["g++", "-std=c++17", "-O1", "-shared", "-fPIC", "-w", "-D__HIP_PLATFORM_AMD__",
                    "-I/opt/rocm/include", os.path.join(HERE, "mock_hip.cpp"), "-o", so], check=True)
    return so


def run(so, code):
    """Output of ``code`` in a child process; the child's failure is the test's."""
    env = dict(os.environ, MOCK_HIP=so, PYTHONPATH=ROOT)
    r = subprocess.run([sys.executable, "-c", "from tests.mock_hip import *\n" + code], env=env, cwd=ROOT,
                       capture_output=True, text=True, timeout=300)
    assert r.returncode == 0, r.stdout + r.stderr
    return r.stdout


# ---- in the child
def start():
    sys.modules["torch"] = None            # it would bring the real runtime
    mock = ctypes.CDLL(os.environ["MOCK_HIP"], ctypes.RTLD_GLOBAL)
    mock.mock_log.restype = mock.mock_stream.restype = ctypes.c_char_p
    mock.mock_bytes.restype = ctypes.c_longlong
    mock.mock_stream.argtypes = [ctypes.c_void_p]
    mock.mock_capture.argtypes = [ctypes.c_void_p, ctypes.c_int]
    return mock


def engine(mol, basis, prepare=True, **kw):
    """An engine whose Schwarz bounds fall with the distance of the shells, so
    that nothing is computed; every class has quartets."""
    import numpy as np
    from quick_amd import basis as B
    from quick_amd.engine import FockEngine
    bs = B.build_basis(mol, basis)
    at = np.array([mol.xyz[s.atom] for s in bs.shells])
    Y = np.exp(-2.0 * np.linalg.norm(at[:, None] - at[None], axis=2))
    e = FockEngine(bs, schwarz=(Y, np.ones((bs.nprim,) * 2)), **kw)
    if prepare:
        e.prepare()
    return e


def launches(mock):
    """The launches since the last mock_clear(); ``before``: every launch that is
    complete when this one starts."""
    out = []
    for line in mock.mock_log().decode().splitlines():
        f = line.split(" ")
        deps = {int(x) for x in f[4:]}
        before = set(deps)
        for d in deps:
            before |= out[d].before
        out.append(Launch(f[1], int(f[2]), int(f[3]), deps, before))
    return out


def slice_doubles(name):
    """Doubles of global slots per workgroup of a recorded kernel (0: none)."""
    m = re.search(r"fused_coop_kernelILb\dELi(\d+)E", name) or re.search(r"fused_grad_coop_kernelILi(\d+)E", name)
    out = []
    for cls, kind in re.findall(r"C(\d{4})(Coop|Grad)E", name):
        with open(os.path.join(ROOT, "quick_amd", "csrc", "gen", ("coop_C" if kind == "Coop" else "grad_C") + cls + ".h")) as f:
            src = f.read()
        src = src[src.index("struct C%s%s" % (cls, kind)):]
        if re.search(r"GLOBAL_SLOTS = (\w+)", src).group(1) in ("true", "1"):
            out.append(int(re.search(r"\bLDS = (\d+)", src).group(1)))
    if not out:
        return 0
    return int(m.group(1)) if m else max(out)
