"""The sweeps with 16, 8 and 4 lanes per atom and with one thread per atom, at the sizes where the
form changes and where the last wave is ragged: the same bits from every form, and the pair force
against the host's serial loop."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _run(tmp_path, cells, species, density, force, pka=0.0, steps=5):
    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / f"{species}.beta")
    names = inputs.workload_beta(path, species)
    md = ea.MD(cells, ntypes=species, seed=11, T=300.0, disp_sigma=0.0 if pka else 0.05, pka_eV=pka)
    inf = md.info()
    fix = ea.FixEPH(inputs.fix_args(path, names, seed=5, flags="7", grid=(cells,) * 3), species,
                    inf["boxlo"], inf["boxhi"], 2.5e-4 if pka else 1e-3, inputs.BOLTZ, inputs.FTM2V,
                    masses=[inputs.MASS_CU] * species)
    fix.init()
    fix.set_sweep_forms(density, force)
    md.attach(fix)
    md.run(fix, steps)
    out = fix.dev_atoms() + (fix.grid().get("T"), fix.get("rho"), fix.get("w"), fix.get("nactive"))
    stats = fix.candidate_stats()
    md.close()
    fix.close()
    return out, stats


# density: 16 lanes up to 8192 atoms, 4 up to 400,000; force: 16 up to 20,000, 8 up to 50,000
@pytest.mark.parametrize("cells,species", [(4, 1), (5, 4), (12, 4), (13, 1), (17, 4), (18, 1), (23, 4),
                                           (24, 1), (46, 1), (47, 4)])
def test_lanes_per_atom_keep_bits(tmp_path, cells, species):
    a, sa = _run(tmp_path, cells, species, "chunk", "chunk")
    b, sb = _run(tmp_path, cells, species, "chunk4", "chunk3")
    for p, q in zip(a, b):
        assert np.array_equal(p, q)
    assert sa == sb


# a fast atom: the waves near it scan their full lists, the lists are rebuilt on the way
@pytest.mark.parametrize("cells", [8, 13])
def test_lanes_per_atom_with_moved_atoms(tmp_path, cells):
    a, sa = _run(tmp_path, cells, 4, "chunk", "chunk", pka=1000.0, steps=25)
    b, sb = _run(tmp_path, cells, 4, "chunk4", "chunk4", pka=1000.0, steps=25)
    for p, q in zip(a, b):
        assert np.array_equal(p, q)
    assert sa == sb


# 16 lanes per atom up to 16,384 atoms, 8 beyond
@pytest.mark.parametrize("cells", [4, 7, 15, 16, 17, 20])
def test_pair_force_matches_host(tmp_path, cells):
    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / "b.beta")
    names = inputs.workload_beta(path, 1)
    md = ea.MD(cells, seed=2, T=300.0, disp_sigma=0.1)
    inf = md.info()
    fix = ea.FixEPH(inputs.fix_args(path, names, grid=(cells,) * 3), 1, inf["boxlo"], inf["boxhi"], 1e-3,
                    inputs.BOLTZ, inputs.FTM2V, masses=[inputs.MASS_CU])
    fix.init()
    s = md.snapshot()
    md.lj(s)
    md.attach(fix)
    assert np.array_equal(fix.dev_atoms()[2], s.f[:s.nlocal])
    md.close()
    fix.close()


# ensembles: ragged chunks, small enough for 16 lanes, for 4 and 8, and beyond
@pytest.mark.parametrize("cells", [(4, 5), (9, 5, 12), (15, 16, 4)])
def test_ensemble_lanes_per_atom_keep_bits(tmp_path, cells):
    import eph_amd as ea
    from eph_amd import inputs
    path = str(tmp_path / "b.beta")
    names = inputs.workload_beta(path, 1)
    out = []
    for form in ("chunk", "chunk4"):
        ens = ea.Ensemble()
        for r, n in enumerate(cells):
            ens.add(dict(cells=n, seed=r + 1, T=300.0, pka_eV=500.0 if n > 8 else 0.0),
                    inputs.fix_args(path, names, seed=r, grid=(n,) * 3), 1, 2.5e-4, inputs.BOLTZ,
                    inputs.FTM2V, [inputs.MASS_CU])
        ens.setup()
        ens.set_variants(form, form)
        ens.run(20)
        out.append([ens.get(r, w) for r in range(len(cells)) for w in ("x", "v", "f", "T", "E")])
        ens.close()
    for p, q in zip(*out):
        assert np.array_equal(p, q)
