"""The audit and the observables of one replica among several, against sums
formed on the host from the downloaded state.  The replicas' colloid counts lie
around the potential kernel's blocks of 32 colloids."""
import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu

COUNTS = (0, 1, 31, 32, 33, 65)
BASE = dict(density=4, n_sub=4, ndt=0.1, kbt=1.0, mass_fl=1.0, mass_colloid=50.0, sig_colloid=3.0, eps=1.0,
            sigma=2.0, theta_deg=90.0, v0=0.05, vel_law=B.BW_VEL_MAXWELL, orient_law=B.BW_ORIENT_SPHERE,
            fluid_init=B.BW_INIT_DEVICE)


def wca(pos, L, sig, eps):
    """(sum, sum of the terms' absolute parts) over pairs i < j, minimum image"""
    i, j = np.triu_indices(len(pos), 1)
    d = pos[i] - pos[j]
    d -= L * np.round(d / L)
    r = np.sqrt((d ** 2).sum(1))
    rc = sig * 2.0 ** (1 / 6)
    fc = 4 * eps * (12 * sig ** 12 / rc ** 13 - 6 * sig ** 6 / rc ** 7)
    ufc = 4 * eps * ((sig / rc) ** 12 - (sig / rc) ** 6) + fc * rc
    r = r[r < rc]
    a, b = 4 * eps * (sig / r) ** 12, 4 * eps * (sig / r) ** 6
    return (a - b - ufc + fc * r).sum(), (a + b + abs(ufc) + abs(fc) * r).sum(), len(r)


@pytest.mark.parametrize("precision", [B.BW_FP64, B.BW_FP32])
def test_audit_and_observables_per_replica(precision):
    e = B.System(replicas=[dict(BASE, L=24, n_colloid=n, seed=50 + n, precision=precision) for n in COUNTS])
    e.startup()
    e.step(2)
    e.observables_reset()
    for r, n in enumerate(COUNTS):
        if n:  # a cubic lattice inside the cutoff, jittered: every colloid has partners
            g = np.stack(np.meshgrid(*[np.arange(5)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
            pos = np.mod(22.0 + 3.1 * g + np.random.default_rng(n).uniform(-0.1, 0.1, (n, 3)), 24.0)
            e.upload_colloid(r, pos=pos)
    e.neighbour_list_md()
    for r, n in enumerate(COUNTS):
        a, o = e.audit(r), e.observables(r)
        _, vel, _ = e.download_fluid(r)
        c = e.download_colloid(r)
        tol = len(vel) * 2.0 ** -52  # FP64 sums of len(vel) terms, in any order
        np.testing.assert_allclose(a["ke_fluid"], 0.5 * (vel ** 2).sum(), rtol=tol)
        np.testing.assert_allclose(a["fluid_momentum"], vel.sum(0), rtol=0, atol=tol * np.abs(vel).sum())
        p = vel.sum(0)
        t_fluid = ((vel ** 2).sum() - (p ** 2).sum() / len(vel)) / (3.0 * (len(vel) - 1))
        np.testing.assert_allclose(o["t_fluid"], t_fluid, rtol=4 * tol)
        if n:
            pot, parts, pairs = wca(c["pos"], 24.0, BASE["sig_colloid"], BASE["eps"])
            assert pairs > 0 or n == 1
            # a term: twelve times the relative error of the distance (one rounding
            # of a coordinate difference below 24, and sqrt), then the sum
            assert abs(a["potential"] - pot) <= (160 + pairs) * 2.0 ** -53 * parts
            np.testing.assert_allclose(o["t_colloid"], 50.0 * (c["vel"] ** 2).sum() / (3.0 * n), rtol=1e-14)
        else:
            assert a["potential"] == 0.0 and o["t_colloid"] == 0.0
