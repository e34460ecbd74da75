"""Clump steps on partner lists against the oracle, which looks for partners in
every step: lists that run out and are built again, bodies too fast for lists
and slow again, more partners than a list holds, bodies that overlap by a face or
by nothing, a loaded state, added and removed bodies, the pairs of a step that
built no tree of its own. Exact."""
import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import clumps as CL

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    L.require_gpu()


def bodies(nb, spacing, v_sigma, seed, static_every=0, spin=0.0):
    s = CL.generate_clumps(seed, nb, spacing=spacing, v_sigma=v_sigma)
    if static_every:
        s["pos4"][::static_every, 3] = 0.0
        for k in ("vel4", "angvel4"):
            s[k][::static_every] = 0.0
    if spin:
        s["angvel4"][:, :3] = np.random.default_rng(seed).normal(0, spin, (nb, 3))
    return s


def compare(sc, o):
    got = sc.download()
    for k, want in (("pos4", o.P), ("vel4", o.V), ("quat4", o.Q), ("angm4", o.L)):
        w = 4 if k == "quat4" else 3
        assert np.array_equal(got[k][:, :w], want[:, :w]), k


def pair_set(p):
    return set(map(tuple, np.asarray(p).tolist()))


# speeds: lists that last long, some steps, none; spacings: few partners, more than a list's 16
@pytest.mark.parametrize("nb,spacing,v,spin", [(1, 0.06, 0.5, 0.0), (2, 0.03, 0.5, 0.0), (63, 0.04, 5.0, 30.0),
                                               (64, 0.04, 0.01, 0.0), (65, 0.035, 30.0, 0.0), (1000, 0.05, 2.0, 100.0),
                                               (1000, 0.05, 20.0, 0.0), (512, 0.05, 120.0, 0.0),
                                               (512, 0.022, 0.3, 0.0)])
def test_lists_run_out(oracle, nb, spacing, v, spin):
    print("[gpu-case] clump lists", nb, spacing, v, spin, flush=True)
    s = bodies(nb, spacing, v, nb, 7 if nb > 100 else 0, spin)
    c = CL.contact_c3()
    o = oracle.ClumpState(s)
    sc = CL.ClumpScene(c)
    sc.upload(s)
    for k in (1, 1, 1, 2, 7, 40, 130, 1):
        sc.step(k)
        o.step(c, k - 1)
        sx, _, lo, hi = o.pose()  # of the last step
        o.step(c, 1)
        compare(sc, o)
        assert pair_set(sc.pairs()) == pair_set(oracle.brute_aabb_pairs(lo, hi))
        assert np.array_equal(sc.spheres(), sx)
        compare(sc, o)
    sc.close()


def test_lists_after_load_add_and_remove(oracle):
    print("[gpu-case] clump lists load", flush=True)
    s, more = bodies(700, 0.045, 3.0, 3), bodies(90, 0.05, 3.0, 4)
    more["pos4"][:, 0] += 0.3
    c = CL.contact_c3()
    o = oracle.ClumpState(s)
    sc = CL.ClumpScene(c)
    sc.upload(s)
    sc.step(25)
    o.step(c, 25)
    buf = sc.save()
    sc.step(33)
    want = sc.download()
    sc.load(buf)  # bodies elsewhere than the lists were built for
    sc.step(33)
    got = sc.download()
    for k in want:
        assert np.array_equal(got[k], want[k]), k
    o.step(c, 33)
    compare(sc, o)
    for act in ("remove", "add", "remove"):
        arg = np.arange(0, o.nb, 9) if act == "remove" else more
        getattr(sc, act)(arg)
        getattr(o, act)(arg)
        sc.step(21)
        o.step(c, 21)
        compare(sc, o)
    stages = sc.profile(5)
    o.step(c, 5)
    compare(sc, o)
    assert stages["partners_contacts"] > 0
    sc.close()


def test_lists_stay_off_without_numbers(oracle):
    """A body that leaves the range of the numbers: its boxes never overlap, the
    others step as before."""
    print("[gpu-case] clump lists overflow", flush=True)
    s = bodies(200, 0.045, 1.0, 8)
    s["vel4"][17, :3] = (3e38, -3e38, 1e30)
    c = CL.contact_c3()
    o = oracle.ClumpState(s)
    sc = CL.ClumpScene(c)
    sc.upload(s)
    for k in (3, 50):
        sc.step(k)
        o.step(c, k)
        got = sc.download()
        rest = np.arange(200) != 17
        for key, want in (("pos4", o.P), ("vel4", o.V), ("quat4", o.Q), ("angm4", o.L)):
            w = 4 if key == "quat4" else 3
            assert np.array_equal(got[key][rest, :w], want[rest, :w]), key
    sc.close()


# slow bodies away from the origin (by so much that rounding takes a part of the
# lists' margin, and all of it), and near it with one far away (a static one)
@pytest.mark.parametrize("off,stray", [(300.0, 0.0), (2500.0, 0.0), (30000.0, 0.0), (0.0, 5000.0), (0.0, 1e6)])
def test_lists_far_from_the_origin(oracle, off, stray):
    print("[gpu-case] clump lists, far", off, stray, flush=True)
    s = bodies(300, 0.09, 0.02, 11)
    s["pos4"][:, 0] += off
    if stray:
        s["pos4"][-1, 1] = stray
        s["pos4"][-1, 3] = 0.0
        s["vel4"][-1] = 0.0
        s["angvel4"][-1] = 0.0
    c = CL.contact_c3()
    o = oracle.ClumpState(s)
    sc = CL.ClumpScene(c)
    sc.upload(s)
    for k in (1, 3, 90, 200):
        sc.step(k)
        o.step(c, k - 1)
        _, _, lo, hi = o.pose()
        o.step(c, 1)
        compare(sc, o)
        assert pair_set(sc.pairs()) == pair_set(oracle.brute_aabb_pairs(lo, hi))
    sc.profile(5)
    o.step(c, 5)
    compare(sc, o)
    sc.close()
