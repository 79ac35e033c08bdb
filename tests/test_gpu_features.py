"""The surrogate's features and range test, whose lanes hold a coarse cell or a
component each: colloid counts around a workgroup's eight, the excluded feature
at the ends of every lane's share."""
import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu

PRM = dict(L=16, density=5, n_sub=5, ndt=0.1, kbt=1.0, mass_fl=1.0, mass_colloid=50.0, sig_colloid=3.0, eps=1.0,
           sigma=2.0, theta_deg=90.0, v0=0.0, seed=3, vel_law=B.BW_VEL_MAXWELL, orient_law=B.BW_ORIENT_SPHERE,
           fluid_init=B.BW_INIT_DEVICE, precision=B.BW_FP64)


@pytest.mark.parametrize("n", [1, 7, 8, 9])
@pytest.mark.parametrize("excluded", [None, 0, 4, 130, 134, 135, 139, 140, 143])
def test_features_and_range(n, excluded):
    s = B.System(n_colloid=n, **PRM)
    s.startup()
    lo, hi = np.full(144, -np.inf, np.float32), np.full(144, np.inf, np.float32)
    if excluded is not None:
        lo[excluded] = np.inf
    s.surrogate_attach(B.MLP(seed=1), lo, hi, np.zeros(6), np.zeros(6))
    s.step(1)  # forms the first moments
    before = s.download_colloid()
    s.step(1)
    assert s.status() == 0
    feat, _, mode = s.surrogate_data()
    assert (mode == (1 if excluded is None else 0)).all()
    np.testing.assert_array_equal(feat[:, 138:141], before["omega"].astype(np.float32))
    np.testing.assert_array_equal(feat[:, 141:144], before["ra"].astype(np.float32))
    np.testing.assert_array_equal(feat[:, 135:138], before["vel"].astype(np.float32))  # v0 = 0: no kick
    dens = feat[:, :135].reshape(n, 27, 5)[:, :, 0] * 8 * PRM["density"]
    # whole particles per coarse cell, within the float32 rounding of n / rho0
    assert np.abs(dens - np.round(dens)).max() <= 2.0 ** -22 * dens.max() and (dens >= 0).all() and dens.max() > 0
