"""GPU: the trajectory gradient where its kernels change form: alpha-table gradients that fit the LDS (2048 knots
in all) or do not, and segments whose steps share the recorded lists between rebuilds."""
import numpy as np
import pytest

from eph_amd.adjoint_worker import build_trajectory

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_beta,nsteps,every", [(64, 12, 12), (64, 20, 10), (2048, 6, 3), (2049, 6, 3)])
def test_beta_gradient_matches_central_differences(tmp_path, n_beta, nsteps, every):
    spec = dict(cells=4, dt=5e-4, nsteps=nsteps, every=every, T=600.0, pka_eV=100.0, target_seed=1, n_beta=n_beta,
                md_seed=7, fix_seed=4711, tmpdir=str(tmp_path))
    md, fix, adj, meta = build_trajectory(spec)
    loss = adj.forward()
    gb, _ = adj.backward()
    b0 = adj.beta0()
    # a smooth direction: the spline's weights are ratios of second differences, which at 2048 knots are some
    # (1 / 2048)^2 = 2e-7 of the values, so that a rough one of h = 1e-6 would leave the linear range
    d = np.cos(np.linspace(0.0, 7.0, b0.size)).reshape(b0.shape) * b0
    h = 1e-6
    fd = (adj.forward(beta=b0 + h * d)[0] - adj.forward(beta=b0 - h * d)[0]) / (2.0 * h)
    ad = float((gb * d).sum())
    # the truncation and rounding of the difference, as for the other gradients
    assert abs(fd - ad) <= 1e-5 * abs(ad) + 1e-9 * abs(loss[0]), (fd, ad)
    adj.close()
