"""Steps on near lists (sd_internal.hpp, StepCtl) against the oracle's search of
every step: lists that run out and are built again, scenes whose spheres are as
wide as their cell (pairs two cells apart can come into contact while a list
lasts), spheres with more contacts than are spread over the wave and more neighbours
than a list holds, static spheres, waves with a few lanes, batches, coordinates far
from the origin, edits and loaded states. Exact."""
import ctypes as C

import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import workloads as W
from stardust_amd.scene import BatchScene, SphereScene

pytestmark = pytest.mark.gpu
COLS = {"x": ("pos4", 0), "y": ("pos4", 1), "z": ("pos4", 2), "vx": ("vel4", 0), "vy": ("vel4", 1), "vz": ("vel4", 2),
        "wx": ("omg4", 0), "wy": ("omg4", 1), "wz": ("omg4", 2)}
MAXC = 64


@pytest.fixture(scope="module", autouse=True)
def gpu():
    L.require_gpu()


def gas(n, r_min, r_max, cell, speed, fill, seed, lo=(0.0, 0.0, 0.0)):
    """Spheres anywhere in a box (overlaps allowed), radii up to half the cell."""
    rng = np.random.default_rng(seed)
    r = rng.uniform(r_min, r_max, n).astype(np.float32)
    r[rng.integers(0, n)] = np.float32(r_max)
    side = float(max(2.0 * cell, (np.sum(4.19 * r.astype(np.float64) ** 3) / fill) ** (1 / 3)))
    lo = np.asarray(lo, np.float64)
    p = (lo + rng.uniform(r_max, max(side - r_max, 1.01 * r_max), (n, 3))).astype(np.float32)
    v = rng.normal(0, speed, (n, 3)).astype(np.float32)
    hi = lo + side
    return p, v, r, W.grid_for(tuple(lo), tuple(hi), cell), (tuple(lo), tuple(hi))


def law(walls, kn=1e3):
    return L.ContactParams.make(kn, 0.3, 0.5, 1e-5, walls=walls, max_contacts=MAXC)


def compare(got, exp, sl=slice(None)):
    for k, (arr, col) in COLS.items():
        assert np.array_equal(got[k][sl], exp[arr][:, col]), k


def run(oracle, p, v, r, m, g, c, calls):
    cols = [np.ascontiguousarray(a) for a in (*p.T, *v.T)]
    sc = SphereScene(g, c, key64=True)
    sc.upload(*cols[:3], r, m, vx=cols[3], vy=cols[4], vz=cols[5])
    st = oracle.SphereState(*cols[:3], r, m, vx=cols[3], vy=cols[4], vz=cols[5], max_contacts=MAXC)
    for k in calls:
        sc.step(k)
        st.step(g, c, nsteps=k, nthreads=8)
        compare(sc.download(), st.by_id())
        assert sc.contact_count() == int(st.hcount.sum())
    sc.close()
    return st


# speeds: lists that last the 64 steps between two looks, some ten steps, a few,
# and none (too fast); one radius: every pair of neighbours across a cell counts
@pytest.mark.parametrize("n,r_min,speed", [(1, 0.01, 1.0), (2, 0.01, 1.0), (63, 0.004, 0.5), (64, 0.01, 0.5),
                                           (65, 0.01, 5.0), (1000, 0.01, 0.05), (3000, 0.01, 2.0), (5000, 0.003, 8.0),
                                           (3000, 0.01, 30.0), (4000, 0.002, 120.0)])
def test_lists_run_out(oracle, n, r_min, speed):
    print("[gpu-case] near lists", n, r_min, speed, flush=True)
    p, v, r, g, walls = gas(n, r_min, 0.01, 0.02, speed, 0.12, n)
    st = run(oracle, p, v, r, W.sphere_mass(r), g, law(walls), (1, 2, 7, 40, 90, 60))
    assert n < 1000 or st.hcount.sum() > 0


# around a large sphere: fewer contacts than are spread over the wave (12), more,
# more neighbours than a list holds (24), many more; the small ones
# cross cells all the time; the large one moving or static
@pytest.mark.parametrize("around,static", [(10, False), (14, False), (17, False), (22, True), (26, False), (45, False), (45, True)])
def test_many_contacts(oracle, around, static):
    print("[gpu-case] many contacts", around, static, flush=True)
    rng = np.random.default_rng(around)
    p, v, r, g, walls = gas(600, 0.003, 0.004, 0.03, 0.3, 0.1, 7)
    big = p[0].copy()
    far = np.linalg.norm(p - big, axis=1) > 0.03
    d = rng.normal(size=(around, 3))
    d /= np.linalg.norm(d, axis=1, keepdims=True)
    p = np.concatenate([[big], big + 0.0174 * d, p[far]]).astype(np.float32)
    r = np.concatenate([[0.015], np.full(around, 0.003), r[far]]).astype(np.float32)
    v = np.concatenate([[[0.0, 0.0, 0.0]], rng.normal(0, 0.2, (around, 3)), v[far]]).astype(np.float32)
    m = W.sphere_mass(r)
    m[0] = 0.0 if static else m[0]
    if static:  # another static sphere in touch: not a contact of two static ones
        m[1] = 0.0
    run(oracle, p, v, r, m, g, law(walls), (1, 3, 30, 70, 300))


def test_batch_of_speeds(oracle):
    """Scenes of other cell sizes, origins and speeds (the margin is the batch's),
    boundaries inside waves."""
    spec = [(700, 0.002, 0.01, 0.3, (0.0, 0.0, 0.0)), (33, 0.01, 0.01, 2.0, (1.0, -2.0, 0.5)),
            (1500, 0.004, 0.012, 1.0, (-3.0, 0.0, 0.0)), (5, 0.005, 0.005, 0.0, (0.0, 4.0, -1.0)),
            (257, 0.006, 0.008, 0.1, (2.0, 2.0, 2.0))]
    parts, states = [], []
    for k, (n, r0, r1, speed, org) in enumerate(spec):
        p, v, r, g, walls = gas(n, r0, r1, 2.0 * r1, speed, 0.12, 50 + k, org)
        c = law(walls, 1e3 * (k + 1))
        cols = [np.ascontiguousarray(a) for a in (*p.T, *v.T)]
        parts.append((n, g, c, cols, r))
        states.append(oracle.SphereState(*cols[:3], r, W.sphere_mass(r), vx=cols[3], vy=cols[4], vz=cols[5],
                                         max_contacts=MAXC))
    cat = [np.concatenate([q[3][a] for q in parts]) for a in range(6)]
    r = np.concatenate([q[4] for q in parts])
    b = BatchScene()
    b.upload_scenes([q[:3] for q in parts], *cat[:3], r, W.sphere_mass(r), vx=cat[3], vy=cat[4], vz=cat[5])
    for steps in (1, 10, 75, 80):
        print("[gpu-case] near lists, batch", steps, flush=True)
        b.step(steps)
        got, off = b.download(), 0
        for (n, g, c, _, _), st in zip(parts, states):
            st.step(g, c, nsteps=steps, nthreads=8)
            compare(got, st.by_id(), slice(off, off + n))
            off += n
    b.close()


def test_edits_and_states_drop_the_lists(oracle):
    """A loaded state, removed and added spheres start from new lists; another law
    keeps them (what bounds them is how far the spheres moved)."""
    p, v, r, g, walls = gas(2000, 0.004, 0.01, 0.02, 0.5, 0.12, 3)
    c = law(walls)
    cols = [np.ascontiguousarray(a) for a in (*p.T, *v.T)]
    sc = SphereScene(g, c, key64=False)
    sc.upload(*cols[:3], r, W.sphere_mass(r), vx=cols[3], vy=cols[4], vz=cols[5])
    st = oracle.SphereState(*cols[:3], r, W.sphere_mass(r), vx=cols[3], vy=cols[4], vz=cols[5], max_contacts=MAXC)
    sc.step(20)
    st.step(g, c, nsteps=20, nthreads=8)
    saved = sc.save()
    sc.step(50)
    sc.load(saved)
    print("[gpu-case] near lists after a load", flush=True)
    sc.step(30)
    st.step(g, c, nsteps=30, nthreads=8)
    compare(sc.download(), st.by_id())
    gone = np.arange(3, 400, 7)
    sc.remove(gone)
    st.remove(gone)
    sc.step(25)
    st.step(g, c, nsteps=25, nthreads=8)
    compare(sc.download(), st.by_id())
    more = [np.ascontiguousarray(a[3:400:7]) for a in cols]
    sc.add(*more[:3], r[3:400:7], W.sphere_mass(r[3:400:7]), vx=more[3], vy=more[4], vz=more[5])
    st.add(*more[:3], r[3:400:7], W.sphere_mass(r[3:400:7]), vx=more[3], vy=more[4], vz=more[5])
    for kn, dt in ((1e3, 1e-5), (4e3, 2e-5), (5e2, 5e-6)):
        c = L.ContactParams.make(kn, 0.2, 0.4, dt, walls=walls, max_contacts=MAXC)
        L.call("sd_ctx_set_contact", sc.h, C.byref(c))
        sc.step(25)
        st.step(g, c, nsteps=25, nthreads=8)
        compare(sc.download(), st.by_id())
    sc.close()


def test_radii_beyond_the_cell(oracle):
    """A loaded state with a sphere wider than its cell keeps no lists (the search
    of 27 cells is the oracle's); the state without it has them again."""
    print("[gpu-case] near lists, radii beyond the cell", flush=True)
    p, v, r, g, walls = gas(2000, 0.004, 0.01, 0.02, 0.5, 0.12, 5)
    c = law(walls)
    cols = [np.ascontiguousarray(a) for a in (*p.T, *v.T)]
    sc = SphereScene(g, c, key64=True)
    sc.upload(*cols[:3], r, W.sphere_mass(r), vx=cols[3], vy=cols[4], vz=cols[5])
    sc.step(20)
    small = sc.save()
    n, head = sc.n, small.nbytes - sc.n * (52 + 8 + 4 + 16 * MAXC)  # header; rows, ids, keys, counts, history
    ids = small[head + 48 * n:head + 52 * n].view(np.int32)

    def oracle_of(buf):
        st = oracle.SphereState(*cols[:3], r, W.sphere_mass(r), max_contacts=MAXC)
        rows = buf[head:head + 48 * n].view(np.float32).reshape(3, n, 4).copy()
        st.pos4, st.vel4, st.omg4, st.ids = rows[0], rows[1], rows[2], ids.copy()
        st.hcount = buf[head + 60 * n:head + 64 * n].view(np.int32).copy()
        st.hist = buf[head + 64 * n:].view(np.float32).reshape(-1, 4).copy()
        return st

    wide = small.copy()
    wide[head:head + 48 * n].view(np.float32).reshape(3, n, 4)[0, ::97, 3] = 0.0137
    for buf in (wide, small, wide):
        sc.load(buf)
        st = oracle_of(buf)
        for k in (1, 30):
            sc.step(k)
            st.step(g, c, nsteps=k, nthreads=8)
            compare(sc.download(), st.by_id())
    sc.close()


# coordinates whose rounding is a thousandth of a radius and more; a grid of more
# than 65,536 cells a side, where every pair's cells are looked at
@pytest.mark.parametrize("off,nx", [(4000.0, 0), (65000.0, 0), (1300.0, 70000)])
def test_lists_far_from_the_origin(oracle, off, nx):
    print("[gpu-case] near lists, far from the origin", off, nx, flush=True)
    cell = 0.02 if nx else 0.5
    lo = (off, -0.5 * off if not nx else 0.0, 0.0)
    p, v, r, g, walls = gas(2000, 0.4 * cell, 0.5 * cell, cell, 20.0, 0.12, 9, lo)
    if nx:
        hi = (nx * cell, *walls[1][1:])
        walls = ((0.0, 0.0, 0.0), hi)
        g = L.Grid.make((0.0, 0.0, 0.0), cell, (nx, *[max(1, int(np.ceil(a / cell))) for a in hi[1:]]))
    r = np.minimum(r, np.float32(0.5 * cell))
    run(oracle, p, v, r, W.sphere_mass(r), g, law(walls), (1, 2, 40, 90))
