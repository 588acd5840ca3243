"""GPU: the forms that a batch's deposit and T_e solve take by the atoms and cells of its replicas, against
separate runs of each replica, bit for bit."""
import numpy as np
import pytest

import eph_amd as ea
from eph_amd import inputs
from drive import workload_files
from test_gpu_ensemble import A, _ensemble, _separate

pytestmark = pytest.mark.gpu


# deposit: a wave per cell (38 atoms per cell on average), counted (378), a thread per cell; solve: one material
# in 4096 and 4097+ cells, per-cell materials in 1728 and 2197; no solve, no random part, no kick; odd and even
# numbers of sub-steps that go through both buffers
@pytest.mark.parametrize("cells,grids,flags,file", [
    ((4, 4), (17, 17), "7", False), ((4, 5), (17, 18), "7", 18), ((4, 5), (17, 18), "7", 19),
    ((4, 5), (17, 18), "7", 20),
    ((4, 5, 6), (2, 2, 3), "7", True), ((4, 5), (1, 1), "7", False), ((4, 5), (17, 6), "7", False),
    ((4, 6), (16, 3), "7", False), ((4, 5), (12, 2), "7", "mixed"), ((4, 5), (13, 6), "7", "mixed"),
    ((4, 5), (9, 6), "7", "mixed"),
    ((4, 5), (4, 4), "3", True), ((4, 5), (4, 4), "5", True), ((4, 5), (4, 4), "6", True),
    ((4, 5), (4, 4), "15", True)])
@pytest.mark.parametrize("graph", [True, False])
def test_batch_forms_match_separate_runs(tmp_path, cells, grids, flags, file, graph):
    species, dt, nsteps = 1, 5e-4, 12
    reps = []
    for k, (n, g) in enumerate(zip(cells, grids)):
        beta, names, tin = workload_files(str(tmp_path), f"r{k}", species, n, A, g, hot_spot=(2000.0, 4.0),
                                          steps=int(file) if isinstance(file, int) and file else 1)
        if file == "mixed":  # another kappa in every third cell
            lines = open(tin).read().split("\n")
            lines[8::3] = [ln.replace(" 0.1 1 0", " 0.05 1 0") for ln in lines[8::3]]
            assert " 0.05 1 0" in lines[8]
            open(tin, "w").write("\n".join(lines))
        if k > 0:
            beta = reps[0][1][16]
        kw = dict(T_infile=tin) if file else {}
        args = inputs.fix_args(beta, names, seed=40 + k, flags=flags, grid=(g, g, g), **kw)
        reps.append((dict(cells=n, a=A, ntypes=species, seed=20 + k, T=900.0, pka_eV=200.0), args))
    ens = _ensemble(reps, species, dt)
    rebuilt = ens.run(nsteps // 2, graph=graph)["rebuilt"]
    rebuilt = np.concatenate([rebuilt, ens.run(nsteps - nsteps // 2, graph=graph)["rebuilt"]])
    for r, (kw, args) in enumerate(reps):
        md, fix = _separate(kw, args, species, dt, rebuilt)
        n = ens.info(r)["nlocal"]
        xs, vs, _ = fix.dev_atoms()
        assert np.array_equal(ens.get(r, "x"), xs[:n]) and np.array_equal(ens.get(r, "v"), vs[:n])
        assert np.array_equal(ens.get(r, "T"), fix.grid().get("T"))
        assert ens.get(r, "E")[1] == fix.compute_vector(0)


# grids finer than the lattice planes: 64 atoms in each of 512 cells and none in most (3 a cell on average), so the
# first deposits are crowded and the next counted ones; the planes then spread and the buckets serve again
@pytest.mark.parametrize("graph", [True, False])
def test_batch_deposit_through_crowded_steps(tmp_path, graph):
    beta, names, _ = workload_files(str(tmp_path), "c", 1, 8, A, 4)
    reps = [(dict(cells=8, a=A, ntypes=1, seed=30 + r, T=2000.0),
             inputs.fix_args(beta, names, seed=50 + r, flags="7", grid=(400, 2, 1), kappa=1e-7)) for r in range(16)]
    ens = _ensemble(reps, 1, 5e-4)
    rebuilt = np.concatenate([ens.run(n, graph=graph)["rebuilt"] for n in (2, 8, 30, 30)])
    for r, (kw, args) in enumerate(reps):
        md, fix = _separate(kw, args, 1, 5e-4, rebuilt)
        xs, vs, _ = fix.dev_atoms()
        n = ens.info(r)["nlocal"]
        assert np.array_equal(ens.get(r, "x"), xs[:n]) and np.array_equal(ens.get(r, "v"), vs[:n])
        assert np.array_equal(ens.get(r, "T"), fix.grid().get("T"))
        assert ens.get(r, "E")[1] == fix.compute_vector(0)
