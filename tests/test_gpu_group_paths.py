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


def sheet(k, n=None):
    """k x k colloids that touch almost (linked into one group)"""
    g = np.stack(np.meshgrid(np.arange(k), np.arange(k), indexing="ij"), -1).reshape(-1, 2)[:n]
    return np.concatenate([3.0 + 5.0 * g, np.full((len(g), 1), 10.0)], 1)


def lattice(n, spacing, origin=(2.0, 2.0, 2.0)):
    k = int(np.ceil(n ** (1 / 3)))
    g = np.stack(np.meshgrid(*[np.arange(k)] * 3, indexing="ij"), -1).reshape(-1, 3)[:n]
    return np.asarray(origin) + spacing * g


def test_cluster_beyond_a_group():
    """100 colloids in one cluster: such a step is taken kernel by kernel, and
    soon only a few are tried by groups first (the tries 1, 3, 7, 15, ...)."""
    a = both(lambda s: place(s, sheet(10)), (3, 12, 5), L=64, n_colloid=100)
    assert a.step_paths() == dict(groups=0, again=4, per_substep=16)


def test_groups_come_back():
    """a cluster, then the same colloids far apart: steps by groups again"""
    far = lattice(36, 13.0)

    def prepare(s):
        place(s, sheet(6))
        s.step(4)
        place(s, far)

    a = both(prepare, (30, 10), L=52, n_colloid=36)
    p = a.step_paths()
    assert p["again"] == 2 and p["per_substep"] <= 5 and p["groups"] >= 37


def test_a_new_start_forgets_clusters():
    s = B.System(**BASE, L=40, n_colloid=36)
    for n in (20, 0):
        s.startup()
        place(s, sheet(6))
        s.step(n)
    p = s.step_paths()
    s.startup()
    place(s, lattice(36, 10.0))
    s.step(5)
    q = s.step_paths()
    assert q["groups"] == p["groups"] + 5 and q["again"] == p["again"] and q["per_substep"] == p["per_substep"]


CROWDED = {
    # events of a substep: about 240 against a list of 128
    "events": (dict(L=40, n_colloid=24, n_sub=1, density=5), lambda: lattice(24, 5.0)),
    # two colloids almost in one place (no forces): their particles are met by both, about 120 against a list of 16
    "shared": (dict(L=40, n_colloid=24, n_sub=1, density=5, eps=0.0),
               lambda: np.concatenate([lattice(12, 5.0), lattice(12, 5.0) + 0.2])),
}


@pytest.mark.parametrize("case", list(CROWDED))
def test_lists_of_a_group_full(case):
    prm, pos = CROWDED[case]
    p = both(lambda s: place(s, pos()), (1,), **prm).step_paths()
    assert p == dict(groups=0, again=1, per_substep=0)


def test_more_events_of_a_colloid_than_its_bucket():
    """Fluid inside a colloid, 64 to 128 events of it in a substep: the
    per-substep kernels replay them serially, in another order of the sums."""
    pos = np.array([[8.3, 8.1, 7.9]])

    def put(s):
        z = np.zeros_like(pos)
        s.upload_colloid(pos=pos, vel=z, omega=z, f=z, old_f=z)

    p = both(put, (1, 2), L=16, n_colloid=1, density=3, mass_colloid=654.1).step_paths()
    assert p["again"] >= 1


def test_small_groups_stay_by_groups():
    p = both(lambda s: place(s, sheet(5, 24)), (2, 3), L=40, n_colloid=24).step_paths()
    assert p == dict(groups=5, again=0, per_substep=0)


def test_full_buckets():
    """Fluid that drifts by two cells a step past heavy colloids: more than
    65536 particles beyond the colloids' buckets."""
    def prepare(s):
        p, v, _ = s.download_fluid()
        s.upload_fluid(p, v + np.array([20.0, 0, 0]))

    p = both(prepare, (1, 1), L=48, n_colloid=100, mass_colloid=1e7).step_paths()
    assert p["groups"] == 0 and p["again"] >= 1


def spinning(neighbours, twice=1, steps=(1,), speed=9.0):
    """A colloid (twice: two of them almost in one place, no forces) that spins
    fast between neighbours just beyond the linking distance: a particle that it
    reflects may come to one of them."""
    c, e = np.array([10.0, 10, 10]), 5.45
    around = np.array([[1.0, 0, 0], [-1, 0, 0], [0, 1, 0], [0, -1, 0]])[:neighbours]
    pos = np.concatenate([[c, c + [0, 0, 0.1]][:twice], c + e * around])
    omega = np.zeros_like(pos)
    omega[:twice, 2] = speed
    return both(lambda s: place(s, pos, omega), steps, L=20, n_colloid=len(pos), density=20, mass_colloid=1e4,
                eps=1.0 if twice == 1 else 0.0)


@pytest.mark.parametrize("twice", [1, 2])
def test_reflected_particle_that_may_reach_another_group(twice):
    assert spinning(4, twice).step_paths() == dict(groups=0, again=1, per_substep=0)


def test_fast_reflected_particle_alone():
    assert spinning(0).step_paths() == dict(groups=1, again=0, per_substep=0)


def test_stopped_steps_among_others():
    """some of the steps of one call are stopped, with steps by groups before and behind them"""
    p = spinning(4, steps=(1, 12, 1, 1, 6), speed=7.5).step_paths()
    assert p["groups"] >= 4 and p["again"] >= 2 and sum(p.values()) == 21


CLUSTER = dict(L=32, n_colloid=25, n_sub=4, density=5)  # beyond a group: every step is stopped


@pytest.mark.parametrize("read", ["status", "audit", "observables", "md_list", "run_counts", "near_particles", "updown"])
def test_reads_behind_a_stopped_step(read):
    """the same as when the steps have been waited for"""
    def result(wait):
        s = B.System(**{**BASE, **CLUSTER})
        s.startup()
        place(s, sheet(5))
        s.neighbour_list_mpcd()
        s.observables_reset()
        s.step(2)
        if wait:
            s.sync()
        if read == "updown":
            s.neighbour_list_mpcd()
            s.updown_velocity()
        r = getattr(s, read)()
        assert s.step_paths()["again"] >= 1
        return r if isinstance(r, dict) else dict(enumerate(r if isinstance(r, tuple) else (r,)))

    a, b = result(False), result(True)
    for k in a:
        np.testing.assert_array_equal(a[k], b[k], err_msg=str(k))


@pytest.mark.parametrize("entry", ["set_v0", "upload_fluid", "upload_colloid", "rotation_mpcd", "run", "update_pos_md",
                                   "update_pos_mpcd", "substep", "set_moments", "profile_steps", "time_steps"])
def test_changes_behind_a_stopped_step(entry):
    def change(s):
        place(s, sheet(5))
        s.step(2)
        if entry == "set_v0":
            s.set_v0(np.full(25, 0.3))
        elif entry == "upload_fluid":
            p, v, _ = s.download_fluid()
            s.step(1)
            s.upload_fluid(p, v)
        elif entry == "upload_colloid":
            s.upload_colloid(vel=np.full((25, 3), 0.1))
        elif entry in ("profile_steps", "time_steps"):
            getattr(s, entry)(3)
        else:
            getattr(s, entry)()

    both(change, (2,), **CLUSTER)


def test_injected_draws_in_a_stopped_step():
    import oracle as O
    from tests.parity import compare_state, inject_step, oracle_step_draws
    prm = dict(L=30, density=5, n_colloid=25, sig_colloid=4.2, sigma=4.0, mass_colloid=50.0, n_sub=4, v0=0.01, theta_deg=90.0, seed=99)
    s = B.System(precision=B.BW_FP64, draws=B.BW_DRAWS_INJECTED, **prm)
    s.startup()
    place(s, sheet(5))
    o = O.Oracle(**prm)
    o.startup()
    o.set_fluid(*s.download_fluid()[:2])
    o.set_colloid(**s.download_colloid())
    o.neighbour_list_mpcd()
    o.neighbour_list_md()
    for _ in range(2):
        shift, axes, refl = oracle_step_draws(o, prm["n_sub"])
        inject_step(s, shift, axes, refl)
        s.step(1)
        assert s.status() == 0
        compare_state(s, o, prm["L"], 1e-10, 1e-10, 1e-10)
    assert s.step_paths()["again"] >= 1


def attach_random_network(s, driven=0.0):
    """drives the colloids whose orientation's x is above `driven`, from the second step on"""
    rng = np.random.default_rng(8)
    net = B.MLP(1)
    net.set_params((0.05 * rng.standard_normal(net.n_params)).astype(np.float32))
    lo, hi = np.full(144, -1e30), np.full(144, 1e30)
    lo[141] = driven
    s.surrogate_attach(net, lo, hi, np.full(6, -20.0), np.full(6, 20.0))
    s.step(1)


@pytest.mark.parametrize("colloids", [24, 25])
def test_driven_and_explicit_colloids_in_one_group(colloids):
    """The surrogate drives about half of a cluster's colloids: in one group (24), in a stopped step (25)."""
    def attach(s):
        place(s, sheet(5, colloids))
        attach_random_network(s)

    s = both(attach, (1, 3), L=32, n_colloid=colloids, n_sub=10, v0=0.03)
    _, imp, mode = s.surrogate_data()
    assert 0 < mode.sum() < colloids and np.abs(imp).sum() > 0
    p = s.step_paths()
    assert p["groups"] == 5 if colloids == 24 else p["again"] >= 2


def test_driven_colloids_with_thin_shells():
    """Shells of about 19 particles: some are too thin for the torque (fewer than
    16), some for the impulse (8), and the colloid takes the mirrored fluid's back."""
    s = both(lambda s: attach_random_network(s, -2.0), (1, 5, 2), L=24, n_colloid=40, n_sub=6, density=1, v0=0.2, sigma=3.0,
             sig_colloid=3.15)
    count, _ = s.surrogate_shells()
    assert (count < 16).any() and s.step_paths()["groups"] == 9


def test_more_colloids_than_the_lists_in_lds():
    """k_group_lists beyond 3072 colloids"""
    prm = [dict(BASE, density=5, L=16, n_colloid=8, n_sub=2, seed=100 + r) for r in range(400)]
    a, b = (B.System(replicas=[dict(p, streaming=v) for p in prm]) for v in (B.BW_STREAM_BLOCKED, B.BW_STREAM_PER_SUBSTEP))
    for s in (a, b):
        s.startup()
        s.step(2)
        assert s.status() == 0
    assert a.step_paths() == dict(groups=2, again=0, per_substep=0)
    for r in range(0, 400, 57):
        ca, cb = a.download_colloid(r), b.download_colloid(r)
        for k in ca:
            np.testing.assert_array_equal(ca[k], cb[k], err_msg=k)
        for x, y in zip(a.download_fluid(r), b.download_fluid(r)):
            np.testing.assert_array_equal(x, y)


def test_more_steps_than_the_list_of_launched_ones():
    """8192 steps may be launched before they are looked at"""
    a, b = (B.System(**{**BASE, "L": 8, "n_colloid": 1, "n_sub": 2, "density": 2, "streaming": v})
            for v in (B.BW_STREAM_BLOCKED, B.BW_STREAM_PER_SUBSTEP))
    for s in (a, b):
        s.startup()
        s.step(8200)
        for _ in range(30):
            s.step(1)
        assert s.status() == 0
    assert a.step_paths()["groups"] == 8230
    for x, y in zip(state(a).values(), state(b).values()):
        np.testing.assert_array_equal(x, y)
