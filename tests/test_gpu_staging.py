"""Downloads around the sizes where the transfer changes: one kernel into the
pinned buffer up to 2 MB in all, pieces of 2 MB and one to eight threads above.
The state that was uploaded comes back, from several threads at once too."""
from concurrent.futures import ThreadPoolExecutor

import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu

BASE = dict(n_sub=4, ndt=0.1, kbt=1.0, mass_fl=1.0, mass_colloid=50.0, sig_colloid=3.0, eps=1.0, sigma=2.0,
            theta_deg=90.0, v0=0.05, seed=7, vel_law=B.BW_VEL_MAXWELL, orient_law=B.BW_ORIENT_SPHERE,
            fluid_init=B.BW_INIT_DEVICE, precision=B.BW_FP64)


# particles x 52 bytes: 27 KB, 1.9 MB (kernel), 2.2 MB (one thread), 14 MB (three), 85 MB (eight)
@pytest.mark.parametrize("L,density", [(8, 1), (16, 9), (24, 3), (30, 10), (48, 15)])
def test_fluid_comes_back(L, density):
    s = B.System(L=L, density=density, n_colloid=0, **BASE)
    s.startup()
    n = L ** 3 * density
    rng = np.random.default_rng(L)
    pos, vel = rng.uniform(0, L, (n, 3)), rng.normal(size=(n, 3))
    s.upload_fluid(pos, vel)
    for _ in range(2):
        p, v, c = s.download_fluid()
        np.testing.assert_array_equal(v, vel)
        np.testing.assert_allclose(p, pos, rtol=0, atol=2.0 ** -52 * L)  # held as cell and offset
        i = np.minimum(p.astype(np.int64), L - 1)
        np.testing.assert_array_equal(c, i[:, 0] + L * (i[:, 1] + L * i[:, 2]))
    with ThreadPoolExecutor(3) as pool:
        for q in pool.map(lambda _: s.download_fluid(), range(3)):
            np.testing.assert_array_equal(q[0], p)
            np.testing.assert_array_equal(q[1], vel)


def test_colloids_come_back():
    s = B.System(replicas=[dict(BASE, L=16, density=1, n_colloid=n) for n in (0, 1, 20)])
    s.startup()
    for r, n in ((1, 1), (2, 20)):
        rng = np.random.default_rng(n)
        sent = {k: rng.uniform(0, 16, (n, 3)) for k in ("pos", "vel", "omega", "f", "old_f", "ra")}
        s.upload_colloid(r, **sent)
        got = s.download_colloid(r)
        for k in sent:
            np.testing.assert_array_equal(got[k], sent[k], err_msg=k)
    assert s.download_colloid(0)["pos"].shape == (0, 3) and s.download_displacement(0).shape == (0, 3)
