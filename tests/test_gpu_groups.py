"""The fused step by colloid groups against the per-substep kernels.

With FP64 storage the two give the same bits for every particle and colloid;
with FP32 storage particles far from every colloid fly in one rounding instead
of n_sub, so after one step velocities and colloid quantities are the same bits
and positions agree to that rounding.  The cases sit where a group's handling
changes: one colloid or several, wrapped boxes, overlapping colloids (serial
replay), clusters and events beyond a group's lists (k_groups_redo), one or few
substeps."""
import numpy as np
import pytest

import brownian_amd as B

pytestmark = pytest.mark.gpu

BASE = dict(density=5, ndt=0.1, kbt=1.0, mass_fl=1.0, mass_colloid=50.0, sig_colloid=4.2, eps=1.0, sigma=4.0,
            theta_deg=90.0, v0=0.05, seed=4321, vel_law=B.BW_VEL_MAXWELL, orient_law=B.BW_ORIENT_SPHERE,
            fluid_init=B.BW_INIT_DEVICE)


def lattice(n, spacing, origin):
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return np.asarray(origin) + spacing * g


# name: parameters, colloid positions to upload after the start-up (None: the start-up's)
CASES = {
    "single": (dict(L=16, n_colloid=1, n_sub=20), None),
    "one_substep": (dict(L=20, n_colloid=4, n_sub=1), None),
    "two_substeps": (dict(L=20, n_colloid=4, n_sub=2), None),
    "odd_substeps": (dict(L=25, n_colloid=9, n_sub=7), None),
    "wrapped_cluster": (dict(L=16, n_colloid=8, n_sub=20), lattice(8, 4.9, (13.0, 13.2, 13.4))),
    "pair_at_the_edge": (dict(L=20, n_colloid=2, n_sub=20), np.array([[19.9, 10.0, 10.0], [4.3, 10.1, 10.0]])),
    "overlapping": (dict(L=20, n_colloid=3, n_sub=20), np.array([[8.0, 10, 10], [11.5, 10, 10.2], [9.7, 13, 10]])),
    "full_group": (dict(L=40, n_colloid=24, n_sub=20), lattice(24, 5.0, (2.0, 2.0, 2.0))),
    "beyond_a_group": (dict(L=40, n_colloid=30, n_sub=10), lattice(30, 5.0, (2.0, 2.0, 2.0))),
    "many_events": (dict(L=16, n_colloid=3, n_sub=5, density=50, mass_colloid=654.1), None),
    "event_lists_full": (dict(L=16, n_colloid=4, n_sub=2, density=30, mass_colloid=654.1),
                         lattice(4, 5.0, (3.0, 3.0, 3.0))),
}


def run(case, precision, streaming, steps):
    prm, pos = CASES[case]
    s = B.System(**{**BASE, **prm, "precision": precision, "streaming": streaming})
    s.startup()
    if pos is not None:
        z = np.zeros_like(pos)
        s.upload_colloid(pos=np.mod(pos, prm["L"]), vel=z, omega=z, f=z, old_f=z)
        fpos, fvel, _ = s.download_fluid()
        d = fpos[:, None] - np.mod(pos, prm["L"])[None]
        d -= prm["L"] * np.round(d / prm["L"])
        inside = ((d ** 2).sum(-1) < 4.41).any(1)  # moved to where another particle is
        free = np.flatnonzero(~inside)
        fpos[inside] = fpos[free[np.arange(inside.sum()) % len(free)]]
        s.upload_fluid(fpos, fvel)
        s.neighbour_list_md()
        s.compute_force_md()
    for n in steps:
        s.step(n)
    flags = s.status(raise_on_error=False)
    fluid = s.download_fluid()
    col = s.download_colloid()
    col["disp"] = s.download_displacement()
    return flags, fluid, col, s.md_list(), s.info[0]["L"]


@pytest.mark.parametrize("case", list(CASES))
def test_groups_equal_per_substep_fp64(case):
    a = run(case, B.BW_FP64, B.BW_STREAM_BLOCKED, (2, 1))
    b = run(case, B.BW_FP64, B.BW_STREAM_PER_SUBSTEP, (2, 1))
    assert a[0] == b[0] == 0
    for x, y in zip(a[1], b[1]):
        np.testing.assert_array_equal(x, y)
    for k in a[2]:
        np.testing.assert_array_equal(a[2][k], b[2][k], err_msg=k)
    for x, y in zip(a[3], b[3]):
        np.testing.assert_array_equal(x, y)


@pytest.mark.parametrize("case", list(CASES))
def test_groups_equal_per_substep_fp32(case):
    a = run(case, B.BW_FP32, B.BW_STREAM_BLOCKED, (1,))
    b = run(case, B.BW_FP32, B.BW_STREAM_PER_SUBSTEP, (1,))
    assert a[0] == b[0] == 0
    np.testing.assert_array_equal(a[1][1], b[1][1])
    for k in a[2]:
        np.testing.assert_array_equal(a[2][k], b[2][k], err_msg=k)
    d = a[1][0] - b[1][0]
    d -= a[4] * np.round(d / a[4])
    assert np.abs(d).max() <= 25 * 2.0 ** -24  # n_sub roundings of an offset below 1


@pytest.mark.parametrize("replicas", [64, 65])
def test_many_groups_equal_per_substep(replicas):
    """512 colloids and more: a workgroup for every group, one wave for lone colloids"""
    prm = [dict(BASE, L=16, n_colloid=8, n_sub=4, seed=100 + r, precision=B.BW_FP64) for r in range(replicas)]
    a, b = (B.System(replicas=[dict(p, streaming=s) for p in prm]) for s in (B.BW_STREAM_BLOCKED, B.BW_STREAM_PER_SUBSTEP))
    for s in (a, b):
        s.startup()
        s.step(2)
        assert s.status() == 0
    for r in (0, replicas // 2, replicas - 1):
        for x, y in zip(a.download_fluid(r), b.download_fluid(r)):
            np.testing.assert_array_equal(x, y)
        ca, cb = a.download_colloid(r), b.download_colloid(r)
        for k in ca:
            np.testing.assert_array_equal(ca[k], cb[k], err_msg=k)
