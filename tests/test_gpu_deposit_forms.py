"""The ordered per-cell sums of the deposit at the item counts where their form changes (a thread or
a wave per cell, one to four items a lane, a workgroup), bit for bit against the oracle's serial loop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


# items per cell of a 4 x 3 x 2 grid; an average of 6 switches from a thread to a wave per cell
@pytest.mark.parametrize("counts", [
    [0, 1, 2, 5, 16, 17], [5, 6, 7, 0, 30, 11], [63, 64, 65, 66, 1, 0], [127, 128, 129, 130, 3, 64],
    [255, 256, 257, 258, 0, 7], [300, 1000, 8192, 8193, 1, 2], [1, 0, 0, 0, 0, 0]])
def test_cell_sums_match_serial_order(oracle, counts):
    import eph_amd as ea
    box = [0.0, 4.0, 0.0, 3.0, 0.0, 2.0]
    rng = np.random.default_rng(sum(counts))
    cell = np.repeat(np.arange(24), np.resize(counts, 24))
    rng.shuffle(cell)
    x = cell % 4 + rng.uniform(0.01, 0.99, len(cell))
    y = cell // 4 % 3 + rng.uniform(0.01, 0.99, len(cell))
    z = cell // 12 + rng.uniform(0.01, 0.99, len(cell))
    # magnitudes over 12 decades, both signs: any other order of the additions shows
    E = rng.standard_normal(len(cell)) * 10.0 ** rng.uniform(-6, 6, len(cell))
    g = ea.Grid.const(4, 3, 2, box, 300.0, 1e-3, 1.0, 0.1)
    o = oracle.FDM.const(4, 3, 2, box, 300.0, 1e-3, 1.0, 0.1)
    for _ in range(2):
        g.insert_energy(x, y, z, E)
        for k in range(len(cell)):
            o.insert_energy(x[k], y[k], z[k], E[k])
    assert np.array_equal(g.get("dT"), o.get("dT"))


# the fix's own deposit: atoms per grid cell from 0.5 to 256 (a thread per cell, a wave per cell,
# then the counted form), with a hot corner so that cells differ
@pytest.mark.parametrize("cells,grid", [(4, 8), (5, 5), (6, 5), (6, 4), (6, 3), (7, 3), (6, 2), (8, 2),
                                        (4, 1), (5, (2, 7, 3))])
def test_deposit_forms_match_oracle(oracle, tmp_path, cells, grid):
    import copy

    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / "b.beta")
    names = inputs.workload_beta(path, 1)
    dims = grid if isinstance(grid, tuple) else (grid,) * 3
    md = ea.MD(cells, seed=4, T=900.0, disp_sigma=0.2)
    inf = md.info()
    args = inputs.fix_args(path, names, seed=3, flags="7", grid=dims)
    cons = (args, 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V)
    ora = oracle.Fix(*cons, masses=[inputs.MASS_CU])
    gpu = ea.FixEPH(*cons, masses=[inputs.MASS_CU])
    gpu.init()
    a = md.snapshot()
    md.lj(a)
    b = copy.deepcopy(a)
    gpu.set_atoms(b)
    for n in (1, 2):
        for fix, s in ((ora, a), (gpu, b)):
            fix.post_force(s, step=n)
            fix.final_integrate(s)
            fix.end_of_step(s, n)
        assert np.array_equal(a.v[:a.nlocal], b.v[:b.nlocal])
        assert np.array_equal(gpu.grid().get("T"), ora.fdm().get("T"))


# a corner of the box holds all atoms, part of it more: queued cells out of the bucket, out of bucket and chain
# (16 slots a cell), and by a scan (27 cells of 1200 atoms in buckets of 1024); so many, or scans so long, that the
# deposits after the first are counted ones
@pytest.mark.parametrize("cells,n,corner", [(6, 4, 0.5), (20, 24, 0.5), (20, 8, 0.5), (20, 30, 0.5), (20, 30, 0.2),
                                            (20, 10, 0.3), (9, 5, 0.2)])
def test_crowded_cells_match_oracle(oracle, tmp_path, cells, n, corner):
    import copy

    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / "b.beta")
    names = inputs.workload_beta(path, 1)
    md = ea.MD(cells, seed=9, T=900.0)
    inf = md.info()
    args = inputs.fix_args(path, names, seed=3, flags="7", grid=(n, n, n))
    cons = (args, 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V)
    ora = oracle.Fix(*cons, masses=[inputs.MASS_CU])
    gpu = ea.FixEPH(*cons, masses=[inputs.MASS_CU])
    gpu.init()
    a = md.snapshot()
    md.lj(a)
    b = copy.deepcopy(a)
    gpu.set_atoms(b)
    ora.post_force(a, step=1)
    gpu.post_force(b, step=1)
    for s in (a, b):  # the deposit sees these positions only
        s.x[:s.nlocal] = np.random.default_rng(1).uniform(0.0, corner, (s.nlocal, 3)) * inf["boxhi"][0]
        s.x[:300] *= 0.4
    for step in (1, 2, 3):
        ora.end_of_step(a, step)
        gpu.end_of_step(b, step)
        assert np.array_equal(gpu.grid().get("T"), ora.fdm().get("T"))


def _fix_pair(oracle, tmp_path, cells, n):
    import copy

    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / "b.beta")
    names = inputs.workload_beta(path, 1)
    md = ea.MD(cells, seed=9, T=900.0)
    inf = md.info()
    args = inputs.fix_args(path, names, seed=3, flags="7", grid=(n, n, n))
    cons = (args, 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V)
    ora = oracle.Fix(*cons, masses=[inputs.MASS_CU])
    gpu = ea.FixEPH(*cons, masses=[inputs.MASS_CU])
    gpu.init()
    a = md.snapshot()
    md.lj(a)
    b = copy.deepcopy(a)
    gpu.set_atoms(b)
    ora.post_force(a, step=1)
    gpu.post_force(b, step=1)
    return md, ora, gpu, a, b


def _fill_cells(x, n, L, counts, seed):
    """the first atoms of x into some of the n^3 cells, counts[k] of them into the k-th"""
    rng = np.random.default_rng(seed)
    out, at = x.copy(), 0
    for c, m in zip(rng.choice(n ** 3, len(counts), replace=False), counts):
        lo = np.array([c % n, c // n % n, c // n ** 2]) * (L / n)
        out[at:at + m] = lo + rng.uniform(0.02, 0.98, (m, 3)) * (L / n)
        at += m
    return out


# cells that overflow after deposits that left the queue empty, so that the queue is the solve's: inside a one-workgroup
# solve (up to 4096 cells) or by its own launch before the tiles (beyond); up to 6 queued cells and more; their atoms
# out of the bucket (256 slots, 1024 with a wave per cell, 16 above 16,384 cells), out of bucket and chain, by a scan
@pytest.mark.parametrize("cells,n,counts", [
    (8, 8, [17]), (8, 8, [20, 40, 64, 100, 256, 30]), (8, 8, [18] * 7), (8, 8, [25] * 20),
    (10, 9, [257, 300, 319]), (10, 9, [330, 700]), (10, 9, [40, 260, 900, 25, 17, 16, 33, 34]),
    (10, 8, [260, 1000]), (12, 8, [1025, 1080, 1100]), (12, 8, [270] * 8),
    (12, 17, [17, 40, 300, 900]), (12, 17, [20] * 9), (10, 26, [17, 40, 79, 500]), (10, 16, [20, 300, 500])])
def test_queue_left_to_the_solve_matches_oracle(oracle, tmp_path, cells, n, counts):
    md, ora, gpu, a, b = _fix_pair(oracle, tmp_path, cells, n)
    L, nl = md.info()["boxhi"][0], a.nlocal
    calm = a.x[:nl].copy()
    step = 0
    for x in (calm, calm, "fill", "fill", calm, calm, "fill"):
        step += 1
        for s in (a, b):  # the deposit sees these positions only
            s.x[:nl] = _fill_cells(calm, n, L, counts, step) if isinstance(x, str) else x
        ora.end_of_step(a, step)
        gpu.end_of_step(b, step)
        assert np.array_equal(gpu.grid().get("T"), ora.fdm().get("T"))
        assert gpu.compute_vector(0) == pytest.approx(ora.compute_vector(0), rel=1e-12)


def _forms(md, fix, steps):
    """in how many of the harness's steps the deposit was bucketed (it then takes the final kick along)"""
    fix.timing(True)
    md.run(fix, steps)
    report = fix.timing_report()
    fix.timing(False)
    return report.get("final_integrate+deposit", (0.0, 0))[1]


# a crowded deposit (900 cells past their buckets; scans over 32,000 atoms for cells of 400), then atoms that are not:
# the deposit after the first counted one is bucketed again
@pytest.mark.parametrize("n,corner", [(24, 0.5), (30, 0.2)])
def test_buckets_return_after_a_crowded_deposit(oracle, tmp_path, n, corner):
    md, _, gpu, _, b = _fix_pair(oracle, tmp_path, 20, n)
    md.attach(gpu)
    assert _forms(md, gpu, 3) == 3
    x = np.random.default_rng(1).uniform(0.0, corner, (b.nlocal, 3)) * md.info()["boxhi"][0]
    x[:300] *= 0.4
    for step in (1, 2, 3):
        b.x[:b.nlocal] = x
        gpu.end_of_step(b, step)
    md.attach(gpu)
    assert _forms(md, gpu, 3) == 2


# 20 queued cells in a one-workgroup solve do not turn the next deposits to the counted form
def test_a_few_queued_cells_keep_the_buckets(oracle, tmp_path):
    md, _, gpu, a, b = _fix_pair(oracle, tmp_path, 8, 8)
    x = a.x[:a.nlocal].copy()
    for step in (1, 2, 3):
        b.x[:b.nlocal] = x if step < 3 else _fill_cells(x, 8, md.info()["boxhi"][0], [25] * 20, 1)
        gpu.end_of_step(b, step)
    md.attach(gpu)
    assert _forms(md, gpu, 2) == 2
