"""Scenes whose lists find no memory, or whose bodies are attached: they hold none
and step by the search of every step, with the same results."""
import ctypes as C
import os
import subprocess
import sys

import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import clumps as CL
from stardust_amd import hullbody as HB
from stardust_amd import hulls as H
from stardust_amd import workloads as W
from stardust_amd.scene import BatchScene, SphereScene

pytestmark = pytest.mark.gpu
ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))

# hipMalloc that finds no memory for sizes within a range
SHIM = r"""
#include <dlfcn.h>
#include <cstdio>
#include <cstdlib>
extern "C" int hipMalloc(void** p, size_t n) {
    using fn = int (*)(void**, size_t);
    static fn real = (fn)dlsym(dlopen("libamdhip64.so.7", RTLD_LAZY | RTLD_LOCAL), "hipMalloc");
    static const size_t lo = strtoull(getenv("REFUSE_FROM"), nullptr, 10), hi = strtoull(getenv("REFUSE_TO"), nullptr, 10);
    if (n >= lo && n <= hi) {
        fprintf(stderr, "refused %zu\n", n);
        *p = nullptr;
        return 2;  // out of memory
    }
    return real(p, n);
}
"""
CHILD = r"""
import ctypes, sys
ctypes.CDLL(sys.argv[1], mode=ctypes.RTLD_GLOBAL)  # before the library that calls it
sys.path.insert(0, sys.argv[2])
from tests import test_gpu_list_memory as T
import numpy as np
np.save(sys.argv[4], getattr(T, sys.argv[3])())
"""
N, NB = 20000, 20000


@pytest.fixture(scope="module", autouse=True)
def gpu():
    L.require_gpu()


def spheres(n=N, seed=4):
    rng = np.random.default_rng(seed)
    cell, m = 0.02, int(np.ceil(n ** (1 / 3)))
    i = rng.permutation(m ** 3)[:n]
    p = ((np.stack([i % m, (i // m) % m, i // (m * m)], 1) + rng.uniform(0.35, 0.65, (n, 3))) * cell).astype(np.float32)
    r = rng.uniform(0.004, 0.0095, n).astype(np.float32)
    v = rng.normal(0, 0.5, (n, 3)).astype(np.float32)
    hi = (m * cell,) * 3
    g = W.grid_for((0, 0, 0), hi, cell)
    c = L.ContactParams.make(1e4, 0.3, 0.5, 1e-5, walls=((0, 0, 0), hi), max_contacts=5)
    return g, c, [np.ascontiguousarray(a) for a in (*p.T, *v.T)], r


def run_spheres():
    g, c, q, r = spheres()
    sc = SphereScene(g, c, key64=True)
    sc.upload(*q[:3], r, W.sphere_mass(r), vx=q[3], vy=q[4], vz=q[5])
    sc.step(60)
    sc.profile(3)
    out = sc.download()
    sc.close()
    return np.stack([out[k] for k in sorted(out)])


def run_clumps():
    s = CL.generate_clumps(5, NB, spacing=0.09, v_sigma=0.2)
    sc = CL.ClumpScene(CL.contact_c3())
    sc.upload(s)
    sc.step(60)
    sc.profile(3)
    out = sc.download()
    out = np.concatenate([out[k] for k in ("pos4", "vel4", "quat4", "angm4")])
    sc.close()
    return out


# the lists are the one allocation of a scene of few stored contacts that takes
# 90 bytes a sphere and more; of a clump scene, 97 bytes a body (its pairs: 96 and 8 KB)
@pytest.mark.parametrize("what,lo,hi", [("run_spheres", 90 * N, 1 << 40), ("run_clumps", 97 * NB, 97 * NB + 64)])
def test_steps_without_memory_for_lists(tmp_path, what, lo, hi):
    print("[gpu-case] no memory for lists", what, flush=True)
    (tmp_path / "shim.cpp").write_text(SHIM)
    (tmp_path / "child.py").write_text(CHILD)
    subprocess.run(["g++", "-O1", "-fPIC", "-shared", str(tmp_path / "shim.cpp"), "-o", str(tmp_path / "shim.so"),
                    "-ldl"], check=True)
    env = dict(os.environ, REFUSE_FROM=str(lo), REFUSE_TO=str(hi))
    r = subprocess.run([sys.executable, str(tmp_path / "child.py"), str(tmp_path / "shim.so"), ROOT, what,
                        str(tmp_path / "out.npy")], env=env, cwd=ROOT, capture_output=True, text=True, timeout=100)
    assert r.returncode == 0, r.stderr[-2000:]
    assert r.stderr.count("refused") == 1, r.stderr[-2000:]
    assert np.array_equal(np.load(tmp_path / "out.npy"), globals()[what]())


def test_attached_scenes_hold_no_lists():
    """Attaching gives the lists' memory back; detaching brings it, and the lists
    are new ones."""
    print("[gpu-case] lists of attached scenes", flush=True)
    n = 600000
    g, c, q, r = spheres(n)
    b = BatchScene()
    alone = SphereScene(g, c, key64=True)
    m = W.sphere_mass(r)
    b.upload_scenes([(n, g, c)], *q[:3], r, m, vx=q[3], vy=q[4], vz=q[5])
    alone.upload(*q[:3], r, m, vx=q[3], vy=q[4], vz=q[5])
    h = H.generate_hulls(0x4C60, 50, lo=(0.0, 0.0, 0.0), hi=(0.1, 0.1, 0.1), v_sigma=0.3)
    bodies, first = HB.concat([HB.make_bodies(h, 0x4C61)])
    law = L.ContactParams.make(2e4, 0.3, 0.5, 1e-5, gravity=(0.0, 0.0, -9.81), walls=None, max_contacts=5)
    hb = HB.HullBodyScene(law)
    hb.upload(bodies, first)

    hip = C.CDLL("libamdhip64.so.7")  # (the one that the library runs on)

    def free():
        L.synchronize()
        room, total = C.c_size_t(), C.c_size_t()
        assert hip.hipMemGetInfo(C.byref(room), C.byref(total)) == 0
        return room.value

    lists = 198 * n

    def step(k):
        b.step(k)
        alone.step(k)
        x, y = b.download(), alone.download()
        for key in x:
            assert np.array_equal(x[key], y[key]), key

    step(23)  # on lists
    before = free()
    b.attach_hulls(hb)
    assert free() - before > 0.8 * lists
    step(9)
    b.autotune(2)
    step(3)
    b.attach_hulls(None)
    step(40)
    b.attach_hulls(hb)  # and back at once: nothing of the lists is left
    b.attach_hulls(None)
    step(40)
    for x in (b, alone, hb):
        x.close()
