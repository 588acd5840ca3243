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
