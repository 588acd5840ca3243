"""The T_e solve's kernel forms (one workgroup, tiles of three sizes, a launch per sub-step) at the
sizes where the form changes and at ragged ones, bit for bit against the oracle's EPH_FDM::solve."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

H = 3.0
C_E, KAPPA = 3e-6, 0.1


def _pair(oracle, dims, T, h=H):
    import eph_amd as ea
    box = [0.0, h * dims[0], 0.0, h * dims[1], 0.0, h * dims[2]]
    g = ea.Grid.const(*dims, box, 300.0, C_E, 1.0, KAPPA)
    o = oracle.FDM.const(*dims, box, 300.0, C_E, 1.0, KAPPA)
    g.set("T", T)
    o.set_T(T)
    return g, o


def _dt(nsub, h=H):
    return (nsub + 0.5) * 0.4 * C_E * h * h / (3.0 * KAPPA) if nsub > 1 else 0.1 * C_E * h * h / KAPPA


# one workgroup (1, 2 and 4 cells a thread), the three tile sizes and their remainders, dimensions
# below a tile and below its halo
@pytest.mark.parametrize("dims,nsub", [
    ((1, 1, 1), 4), ((3, 1, 2), 3), ((4, 4, 4), 19), ((32, 32, 1), 2), ((31, 11, 3), 5),
    ((16, 16, 16), 7), ((4097, 1, 1), 4), ((17, 16, 16), 1), ((17, 16, 16), 2), ((9, 22, 23), 4),
    ((2, 70, 37), 6), ((41, 40, 39), 19), ((200, 3, 7), 5), ((64, 64, 50), 2), ((67, 63, 59), 5),
    ((80, 64, 80), 3), ((77, 75, 73), 4)])
def test_uniform_grid_forms_match_oracle(oracle, dims, nsub):
    n = dims[0] * dims[1] * dims[2]
    rng = np.random.default_rng(n + nsub)
    g, o = _pair(oracle, dims, 300.0 + 1000.0 * rng.uniform(size=n))
    g.set_dt(_dt(nsub))
    o.set_dt(_dt(nsub))
    for _ in range(2):
        p = rng.uniform(-0.1, 1.1, (3, 40)) * H * np.array(dims)[:, None]
        e = rng.uniform(-1e-3, 1e-3, 40)
        g.insert_energy(*p, e)
        for k in range(40):
            o.insert_energy(p[0, k], p[1, k], p[2, k], e[k])
        assert g.solve() == o.solve() == nsub
        assert np.array_equal(g.get("T"), o.get("T"))
        assert not g.get("dT").any()


# temperatures and deposits that the quotients by a known reciprocal do not cover, from the start or
# from a later sub-step on, in the block and the tile form
@pytest.mark.parametrize("dims", [(6, 5, 4), (20, 19, 17)])
@pytest.mark.parametrize("value", [0.0, 1e-160, 5e-324, 1e160, 1e300])
def test_uniform_grid_extreme_values_match_oracle(oracle, dims, value):
    n = dims[0] * dims[1] * dims[2]
    T = np.full(n, 300.0)
    T[n // 2] = value
    T[1] = 0.0
    g, o = _pair(oracle, dims, T)
    g.set_dt(_dt(5))
    o.set_dt(_dt(5))
    for _ in range(2):
        assert g.solve() == o.solve()
        assert np.array_equal(g.get("T"), o.get("T"))


@pytest.mark.parametrize("h", [1e-3, 2.0 ** -22, 1e9])
def test_uniform_grid_spacings_match_oracle(oracle, h):
    dims = (9, 7, 5)
    rng = np.random.default_rng(3)
    g, o = _pair(oracle, dims, 300.0 + 10.0 * rng.uniform(size=315), h)
    g.set_dt(_dt(3, h))
    o.set_dt(_dt(3, h))
    assert g.solve() == o.solve()
    assert np.array_equal(g.get("T"), o.get("T"))


# values per cell (walls, constant cells, sources, unequal kappa): one workgroup up to 2048 cells,
# one launch per sub-step beyond
@pytest.mark.parametrize("dims", [(4, 4, 4), (16, 16, 8), (16, 16, 9), (5, 33, 3)])
@pytest.mark.parametrize("tdyn", [False, True])
def test_mixed_grid_forms_match_oracle(oracle, tmp_path, dims, tdyn):
    import eph_amd as ea
    from eph_amd import inputs
    n = dims[0] * dims[1] * dims[2]
    rng = np.random.default_rng(n)
    T = 300.0 + 500.0 * rng.uniform(size=n)
    params = str(tmp_path / "p")
    t = np.arange(200) * 20.0
    inputs.write_params(params, 20.0, C_E * (1.0 + t / 3000.0), KAPPA * (1.0 + t / 6000.0))
    path = str(tmp_path / "g")
    inputs.write_grid(path, *dims, [0, H * dims[0], 0, H * dims[1], 0, H * dims[2]], T,
                      S=1e-4 * rng.uniform(size=n) * (rng.uniform(size=n) < 0.2), C_e=C_E,
                      kappa=KAPPA * rng.choice([1.0, 0.5], n), flag=rng.choice([1, 1, 1, 0, 2], n),
                      tdyn=rng.choice([0, 1], n) if tdyn else 0, params=params)
    g, o = ea.Grid.load(path), oracle.FDM.load(path)
    g.set_dt(_dt(6))
    o.set_dt(_dt(6))
    for _ in range(3):
        assert g.solve() == o.solve()
        assert np.array_equal(g.get("T"), o.get("T"))


def test_grid_turns_from_uniform_to_mixed(oracle):
    """a cell set after solves of one material: the per-cell form takes over"""
    dims = (12, 12, 12)
    rng = np.random.default_rng(5)
    g, o = _pair(oracle, dims, 300.0 + 100.0 * rng.uniform(size=1728))
    g.set_dt(_dt(4))
    o.set_dt(_dt(4))
    assert g.solve() == o.solve()
    for x in (g, o):
        x.set_cell(3, 4, 5, 400.0, 1e-4, 1.0, 2 * C_E, 0.5 * KAPPA, 0, 0)
    for _ in range(2):
        assert g.solve() == o.solve()
        assert np.array_equal(g.get("T"), o.get("T"))
