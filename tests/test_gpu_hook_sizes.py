"""GPU: the host-array hooks on both sides of the sizes up to which their arrays go through pinned memory in
place (1 MB of them per hook), bit for bit against the oracle, and the T_e grid's copies likewise."""
import copy

import numpy as np
import pytest

import eph_amd as ea
from eph_amd import inputs
from drive import workload_files

pytestmark = pytest.mark.gpu


# atoms (and ghosts): 108, 864, 4000 small in every hook; 8788 beyond it in initial_integrate and post_force only;
# 13500 in final_integrate too; 23328 in all of them
@pytest.mark.parametrize("cells", [3, 6, 10, 13, 15, 18])
@pytest.mark.parametrize("timed", [False, True])
def test_hooks_match_oracle_at_every_size(oracle, tmp_path, cells, timed):
    if timed and cells > 6:
        pytest.skip("the timed hooks take the same path at every size")
    md = ea.MD(cells, a=3.615, ntypes=2, seed=7, T=600.0, disp_sigma=0.05)
    inf = md.info()
    beta, names, tin = workload_files(str(tmp_path), "h", 2, cells, 3.615, 4, hot_spot=(2000.0, 4.0))
    args = inputs.fix_args(beta, names, seed=5, flags="7", grid=(4, 4, 4), T_infile=tin)
    cons = (args, 2, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V)
    ora = oracle.Fix(*cons, masses=[inputs.MASS_CU] * 2)
    gpu = ea.FixEPH(*cons, masses=[inputs.MASS_CU] * 2)
    gpu.init()
    gpu.timing(timed)
    a = md.snapshot()
    md.lj(a)
    b = copy.deepcopy(a)
    gpu.set_atoms(b)
    for step in (1, 2):
        for fix, s in ((ora, a), (gpu, b)):
            fix.initial_integrate(s)
            md.update_ghosts(s)
            md.lj(s)
            fix.post_force(s, step=step)
            fix.final_integrate(s)
            fix.end_of_step(s, step)
        n = a.nlocal
        assert np.array_equal(a.x[:n], b.x[:n]) and np.array_equal(a.v[:n], b.v[:n])
        assert np.array_equal(a.f[:n], b.f[:n])
        assert np.array_equal(gpu.grid().get("T"), ora.fdm().get("T"))
    x, v, f = gpu.dev_atoms()
    assert np.array_equal(x[:n], a.x[:n]) and np.array_equal(v[:n], a.v[:n]) and np.array_equal(f[:n], a.f[:n])


# points (4 doubles each) and cells (one) around 1 MB
@pytest.mark.parametrize("n", [1, 1000, 32768, 32769])
def test_grid_copies_match_at_every_size(oracle, n):
    box = [0.0, 4.0, 0.0, 3.0, 0.0, 2.0]
    rng = np.random.default_rng(n)
    x, y, z = rng.uniform(0, 4, n), rng.uniform(0, 3, n), rng.uniform(0, 2, n)
    E = rng.standard_normal(n)
    for dims in ((3, 3, 3), (64, 64, 32), (64, 64, 33)):
        g = ea.Grid.const(*dims, box, 300.0, 1e-3, 1.0, 0.1)
        o = oracle.FDM.const(*dims, box, 300.0, 1e-3, 1.0, 0.1)
        g.insert_energy(x, y, z, E)
        for k in range(n):
            o.insert_energy(x[k], y[k], z[k], E[k])
        assert np.array_equal(g.get("dT"), o.get("dT")) and np.array_equal(g.get("T"), o.get("T"))
