"""GPU: a deposit whose buckets find no memory takes the counted form and leaves the same bits.  The allocations are
refused by a hipMalloc of this test's own, in a process of its own, from a size on that only the buckets reach."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = 0;
static int refused = 0;
extern "C" void shim_limit(size_t n) { limit = n; refused = 0; }
extern "C" int shim_refused() { return refused; }
extern "C" int hipMalloc(void** p, size_t n) {
  typedef int (*fn)(void**, size_t);
  static fn real = reinterpret_cast<fn>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc"));
  if (limit && n >= limit) {
    ++refused;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
"""

CHILD = r"""
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library and the runtime are loaded
shim.shim_limit.argtypes = [C.c_size_t]
import numpy as np
import eph_amd as ea
from eph_amd import inputs

names = inputs.workload_beta(sys.argv[2], 1)
cons = dict(seed=3, flags="7", grid=(16, 16, 16))  # buckets of 4.2 MB (8.5 MB for two replicas), all else below 4 MB


def single():
    md = ea.MD(8, seed=9, T=900.0)
    inf = md.info()
    fix = ea.FixEPH(inputs.fix_args(sys.argv[2], names, **cons), 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ,
                    inputs.FTM2V, masses=[inputs.MASS_CU])
    fix.init()
    md.attach(fix)
    md.run(fix, 5)
    return (*fix.dev_atoms(), fix.grid().get("T"), fix.compute_vector(0))


def batch():
    ens = ea.Ensemble()
    for r in range(2):
        ens.add(dict(cells=8, seed=r + 1, T=300.0), inputs.fix_args(sys.argv[2], names, **cons), 1, 1e-3, inputs.BOLTZ,
                inputs.FTM2V, [inputs.MASS_CU])
    ens.setup()
    ens.run(5)
    return [ens.get(r, w) for r in range(2) for w in ("x", "v", "f", "T", "E")]


for f in (single, batch):
    out = []
    for limit in (0, 4 << 20):
        shim.shim_limit(limit)
        out.append(f())
        assert (shim.shim_refused() > 0) == (limit > 0), (f.__name__, limit, shim.shim_refused())
    for a, b in zip(*out):
        assert np.array_equal(a, b), f.__name__
print("same bits")
"""


def test_deposit_without_memory_for_buckets(tmp_path):
    shim = str(tmp_path / "shim.so")
    src = tmp_path / "shim.cpp"
    src.write_text(SHIM)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", shim, str(src), "-ldl"])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=os.path.join(root, "user-eph_amd") + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", CHILD, shim, str(tmp_path / "b.beta")], env=env, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and "same bits" in r.stdout, r.stdout + r.stderr
