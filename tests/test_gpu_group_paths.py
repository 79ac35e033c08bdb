"""The fused step by colloid groups where it leaves its usual way, against the
per-substep kernels: FP64 storage, the same bits for every particle and
colloid, and no status flag."""
import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu

BASE = dict(density=10, n_sub=20, ndt=0.1, kbt=1.0, mass_fl=1.0, mass_colloid=50.0, sig_colloid=4.2, eps=1.0, sigma=4.0,
            theta_deg=90.0, v0=0.0, seed=4321, vel_law=B.BW_VEL_MAXWELL, orient_law=B.BW_ORIENT_SPHERE,
            fluid_init=B.BW_INIT_DEVICE, precision=B.BW_FP64)


def distance(a, b, L):
    d = a - b
    return np.sqrt(((d - L * np.round(d / L)) ** 2).sum(-1))


def place(s, pos, omega=None, edit=None):
    """Colloids at rest at pos, the fluid inside them moved outside at random;
    edit(positions, velocities) of the fluid in place."""
    L = s.info[0]["L"]
    pos = np.mod(pos, L)
    z = np.zeros_like(pos)
    s.upload_colloid(pos=pos, vel=z, omega=z if omega is None else omega, f=z, old_f=z)
    fpos, fvel, _ = s.download_fluid()
    rng = np.random.default_rng(3)
    inside = np.zeros(len(fpos), bool)
    for p in pos:
        inside |= distance(fpos, p, L) < 2.0
    for i in np.flatnonzero(inside):
        while distance(pos, fpos[i], L).min() < 2.0:
            fpos[i] = rng.uniform(0, L, 3)
    if edit is not None:
        edit(fpos, fvel)
    s.upload_fluid(fpos, fvel)
    s.neighbour_list_md()
    s.compute_force_md()


def state(s):
    out = dict(zip(("fluid_pos", "fluid_vel", "fluid_cell"), s.download_fluid()), **s.download_colloid())
    return dict(out, disp=s.download_displacement())


def both(prepare, steps, **params):
    """Final states by groups (the context comes back too) and per substep,
    after the same calls of step; equal, without flags."""
    a, b = (B.System(**{**BASE, **params, "streaming": v}) for v in (B.BW_STREAM_BLOCKED, B.BW_STREAM_PER_SUBSTEP))
    for s in (a, b):
        s.startup()
        prepare(s)
        for n in steps:
            s.step(n)
    assert b.status(raise_on_error=False) == 0
    assert a.status(raise_on_error=False) == 0
    sa, sb = state(a), state(b)
    for k in sa:
        np.testing.assert_array_equal(sa[k], sb[k], err_msg=k)
    return a


def test_chain_across_half_the_box():
    """Colloids linked by fast particles, 9 apart: the group reaches from its
    first colloid past half the box, where a particle and a colloid next to it
    may have their nearest images on different sides."""
    L = 52

    def edit(p, v):
        fast = np.array([[6.5 + 9 * i, 26, 26] for i in range(3)])
        for i, q in enumerate(fast):  # alone in its cell, so that the rotation leaves its velocity
            m = (np.abs(p - q) < 2.2).all(1)
            m[:3] = False
            p[m] = np.random.default_rng(i).uniform([0, 0, 35], [L, L, 50], (m.sum(), 3))
        p[:3] = fast
        v[:3] = [0, 23.0, 0]

    both(lambda s: place(s, np.array([[2.0 + 9 * i, 26, 26] for i in range(4)]), edit=edit), (1,), L=L, n_colloid=4)
