"""GPU: the harness's steps with the small launches folded into their neighbours against the same steps with
every launch of its own, bit for bit."""
import numpy as np
import pytest

import eph_amd as ea
from eph_amd import inputs
from drive import workload_files

pytestmark = pytest.mark.gpu


# one with the check, ghost, flag and tally launches folded into their neighbours, one with each in its own
# launch (as the timing report wants them): NOINT (flag 8), no solve, no deposit, another model's sweeps; the
# fused tally in a one-workgroup solve, in tiles and behind a counted deposit; above the speculated sizes
@pytest.mark.parametrize("cells,grid,flags,model", [
    (6, 6, "7", "4"), (6, 6, "15", "4"), (6, 6, "3", "4"), (6, 6, "4", "4"), (6, 6, "5", "4"),
    (6, 6, "6", "4"), (6, 1, "7", "4"), (6, 2, "7", "4"), (6, 20, "7", "4"), (6, 6, "7", "1"),
    (26, 10, "7", "4"), (26, 26, "7", "4")])
def test_fused_steps_match_separate_launches(tmp_path, cells, grid, flags, model):
    out = []
    for timed in (False, True):
        md = ea.MD(cells, a=3.615, ntypes=1, seed=5, T=300.0, pka_eV=200.0)
        inf = md.info()
        beta, names, tin = workload_files(str(tmp_path), "s", 1, cells, 3.615, grid, None)
        args = inputs.fix_args(beta, names, seed=99, flags=flags, model=model, grid=(grid,) * 3, T_infile=tin)
        fix = ea.FixEPH(args, 1, inf["boxlo"], inf["boxhi"], 1e-3, inputs.BOLTZ, inputs.FTM2V,
                        masses=[inputs.MASS_CU])
        fix.init()
        md.attach(fix)
        fix.timing(timed)
        res = md.run(fix, 15, first_step=1)
        assert res["total_ms"] > 0 and res["fix_ms"] > 0 and res["pair_ms"] > 0
        out.append((res["rebuilds"], *fix.dev_atoms(), fix.grid().get("T"), fix.grid().get("dT"),
                    fix.compute_vector(0)))
    assert out[0][0] == out[1][0] and (out[0][0] > 0 or "15" == flags)
    for a, b in zip(out[0][1:], out[1][1:]):
        assert np.array_equal(a, b)


# atoms pushed together between two runs, so that a rebuild on the device exceeds its list capacity (1.25 times the
# longest list and 16) and the host takes it over: with the pair force queued ahead of the check, and above that size
@pytest.mark.parametrize("cells", [6, 26])
def test_rebuild_beyond_the_capacity_matches_host_rebuild(tmp_path, cells):
    out = []
    for device in (True, False):
        md = ea.MD(cells, a=3.615, ntypes=1, seed=5, T=300.0)
        inf = md.info()
        beta, names, _ = workload_files(str(tmp_path), "o", 1, cells, 3.615, 6)
        args = inputs.fix_args(beta, names, seed=99, flags="7", grid=(6, 6, 6), kappa=0.02)
        fix = ea.FixEPH(args, 1, inf["boxlo"], inf["boxhi"], 1e-4, inputs.BOLTZ, inputs.FTM2V,
                        masses=[inputs.MASS_CU])
        fix.init()
        md.attach(fix)
        md.set_device_rebuild(device)
        md.run(fix, 1)
        s = md.snapshot()
        n = s.nlocal
        x, v, _ = fix.dev_atoms()
        mid = 0.5 * np.asarray(inf["boxhi"])
        s.x[:n], s.v[:n] = mid + 0.85 * (x[:n] - mid), v[:n]
        fix.end_of_step(s, 1)  # (puts the positions on the device)
        md.force_rebuild()
        res = md.run(fix, 3, first_step=2)
        assert res["rebuilds"] >= 1
        longest = np.diff(md.snapshot().nbr_off).max()
        out.append((longest, *fix.dev_atoms(), fix.grid().get("T"), fix.compute_vector(0)))
    assert out[0][0] > 123  # 86 entries at the start, and so a capacity of 123
    for a, b in zip(*out):
        assert np.array_equal(a, b)
