"""GPU: a second thread reads values of a grid or a fix while the first one calls it, both through the pinned
memory of small calls: every value read and every state stepped is the one of calls in turn."""
import threading

import numpy as np
import pytest

import eph_amd as ea
from eph_amd import inputs
from drive import workload_files

pytestmark = pytest.mark.gpu


def _together(work, reader):
    """work() on this thread, reader() again and again on another until it is done"""
    done, errors, reads = threading.Event(), [], [0]

    def loop():
        try:
            while not done.is_set():
                reader()
                reads[0] += 1
        except BaseException as e:  # noqa: BLE001 (reported below)
            errors.append(e)

    t = threading.Thread(target=loop)
    t.start()
    try:
        work()
    finally:
        done.set()
        t.join()
    assert not errors, errors[0]
    assert reads[0] > 0


def test_two_readers_of_one_grid():
    dims, rng = (20, 20, 10), np.random.default_rng(1)
    g = ea.Grid.const(*dims, [0, 60, 0, 60, 0, 30], 300.0, 3e-6, 1.0, 0.1)
    T, kappa = rng.uniform(300, 400, 4000), rng.uniform(0.05, 0.1, 4000)
    g.set("T", T)
    g.set("kappa", kappa)

    def read_T():
        assert np.array_equal(g.get("T"), T)

    def read_kappa():
        for _ in range(400):
            assert np.array_equal(g.get("kappa"), kappa)

    _together(read_kappa, read_T)


def test_values_read_while_a_fix_steps(tmp_path):
    def run(watched):
        md = ea.MD(4, a=3.615, ntypes=1, seed=3, T=600.0, disp_sigma=0.05)
        inf = md.info()
        beta, names, tin = workload_files(str(tmp_path), "t", 1, 4, 3.615, 8, hot_spot=(2000.0, 4.0))
        args = inputs.fix_args(beta, names, seed=5, flags="7", grid=(8, 8, 8), T_infile=tin)
        fix = ea.FixEPH(args, 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V,
                        masses=[inputs.MASS_CU])
        fix.init()
        s = md.snapshot()
        md.lj(s)
        fix.set_atoms(s)
        grid = fix.grid()

        def steps():
            for n in range(1, 61):
                fix.initial_integrate(s)
                md.update_ghosts(s)
                md.lj(s)
                fix.post_force(s, step=n)
                fix.final_integrate(s)
                fix.end_of_step(s, n)

        def read():
            assert 250.0 < grid.get("T").min() and grid.get("T").max() < 2500.0
            assert np.isfinite(fix.compute_vector(0)) and 300.0 < fix.compute_vector(1) < 1000.0

        _together(steps, read if watched else lambda: None)
        return s.x, s.v, s.f, grid.get("T"), fix.compute_vector(0)

    for a, b in zip(run(False), run(True)):
        assert np.array_equal(a, b)
