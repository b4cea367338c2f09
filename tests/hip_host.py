"""Runs code against libsac_amd.so on the HIP runtime of hip_host.c, in a
process of its own (the library's references are bound once per process)."""
import os
import subprocess
import sys
import textwrap

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)

PRELUDE = """
import ctypes, sys
import numpy as np
sys.path.insert(0, {root!r})
hip = ctypes.CDLL({stub!r}, mode=ctypes.RTLD_GLOBAL)
ctypes.CDLL("libstdc++.so.6", mode=ctypes.RTLD_GLOBAL)  # what operator new throws

def knob(name, kind=ctypes.c_int):
    return kind.in_dll(hip, "hip_host_" + name)

from sac_amd import device, batch, problems
from tests.hip_host import state_problem
"""


def state_problem(n, seed=5):
    """A problem of extents n whose variables are all drawn at random."""
    import numpy as np
    from sac_amd import problems
    side = {"rho": 1.0, "p": 1.0, "v": [0, 0, 0], "b": [1, 0, 0]}
    if len(n) == 1:
        prob = problems.riemann_tube(n[0], side, side)
    elif len(n) == 2:
        prob = problems.riemann_patch(*n, side, side)
    else:
        prob = problems.stratified(n=n[0], nxyz=n)
    prob.w = np.random.default_rng(seed).standard_normal(prob.w.shape)
    return prob


def build(folder):
    out = os.path.join(str(folder), "hip_host.so")
    subprocess.run(["gcc", "-O2", "-Wall", "-fexceptions", "-shared", "-fPIC", "-pthread",
                    os.path.join(HERE, "hip_host.c"), "-o", out], check=True)
    return out


def run(stub, code):
    """Run `code` after PRELUDE; its assertions are the test's."""
    src = PRELUDE.format(root=ROOT, stub=stub) + textwrap.dedent(code)
    r = subprocess.run([sys.executable, "-c", src], capture_output=True, text=True, timeout=120,
                       cwd=ROOT)
    assert r.returncode == 0, f"exit {r.returncode}\n{r.stdout}\n{r.stderr}"
