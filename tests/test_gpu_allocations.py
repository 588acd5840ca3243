"""GPU: the library's allocations, seen through a hipMalloc and hipHostMalloc of this test's own in a process of its
own.  A deposit whose buckets find no memory (they are refused from a size on that only the buckets reach) takes the
counted form and leaves the same bits; and the first hooks on new atoms, like the first calls on a new grid, find their
pinned memory and the deposit's buffers made."""
import os
import subprocess
import sys

import pytest

pytestmark = pytest.mark.gpu

SHIM = r"""
#include <dlfcn.h>
#include <stddef.h>
static size_t limit = 0;
static int refused = 0, device = 0, pinned = 0;
extern "C" int shim_device() { return device; }
extern "C" int shim_pinned() { return pinned; }
extern "C" int hipHostMalloc(void** p, size_t n, unsigned flags) {
  typedef int (*fn)(void**, size_t, unsigned);
  static fn real = reinterpret_cast<fn>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipHostMalloc"));
  ++pinned;
  return real(p, n, flags);
}
extern "C" void shim_limit(size_t n) { limit = n; refused = 0; }
extern "C" int shim_refused() { return refused; }
extern "C" int hipMalloc(void** p, size_t n) {
  typedef int (*fn)(void**, size_t);
  static fn real = reinterpret_cast<fn>(dlsym(dlopen("libamdhip64.so.7", RTLD_NOW), "hipMalloc"));
  ++device;
  if (limit && n >= limit) {
    ++refused;
    return 2;  // hipErrorOutOfMemory
  }
  return real(p, n);
}
"""

START = r"""
import ctypes as C, sys
shim = C.CDLL(sys.argv[1], mode=C.RTLD_GLOBAL)  # before the library and the runtime are loaded
shim.shim_limit.argtypes = [C.c_size_t]
import numpy as np
import eph_amd as ea
from eph_amd import inputs

names = inputs.workload_beta(sys.argv[2], 1)
"""

REFUSED = START + r"""
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


FIRST = START + r"""
for cells, grid in ((4, 4), (8, 16), (20, 20), (20, 10)):
    md = ea.MD(cells, seed=9, T=900.0)
    inf = md.info()
    fix = ea.FixEPH(inputs.fix_args(sys.argv[2], names, seed=3, flags="7", grid=(grid,) * 3), 1, inf["boxlo"],
                    inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V, masses=[inputs.MASS_CU])
    fix.init()
    s = md.snapshot()
    md.lj(s)
    fix.set_atoms(s)
    before = shim.shim_device(), shim.shim_pinned()
    assert min(before) > 0
    for n in (1, 2):
        fix.initial_integrate(s)
        fix.post_force(s, step=n)
        fix.final_integrate(s)
        fix.end_of_step(s, n)
        fix.grid().get("T"), fix.compute_vector(0)
    assert (shim.shim_device(), shim.shim_pinned()) == before, (cells, grid, before)
g = ea.Grid.const(21, 17, 24, [0, 63, 0, 51, 0, 72], 300.0, 3e-6, 1.0, 0.1)
before = shim.shim_pinned()
x = np.linspace(0.0, 50.0, 5000)
g.insert_energy(x, x, x, 1e-6 * x)
g.solve(), g.get("T"), g.T_mean()
assert shim.shim_pinned() == before
print("nothing allocated")
"""


def _child(tmp_path, script, says):
    shim = str(tmp_path / "shim.so")
    src = tmp_path / "shim.cpp"
    src.write_text(SHIM)
    subprocess.check_call(["g++", "-O1", "-shared", "-fPIC", "-o", shim, str(src), "-ldl"])
    root = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
    env = dict(os.environ, PYTHONPATH=os.path.join(root, "user-eph_amd") + os.pathsep + os.environ.get("PYTHONPATH", ""))
    r = subprocess.run([sys.executable, "-c", script, shim, str(tmp_path / "b.beta")], env=env, capture_output=True,
                       text=True, timeout=100)
    assert r.returncode == 0 and says in r.stdout, r.stdout + r.stderr


def test_deposit_without_memory_for_buckets(tmp_path):
    _child(tmp_path, REFUSED, "same bits")


def test_first_hooks_allocate_nothing(tmp_path):
    _child(tmp_path, FIRST, "nothing allocated")
