"""Re-sorts of thousands of changed cells (scenes of more than 262,144 spheres
take up to one sphere in 256 per step) against the oracle's full sort. Exact."""
import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import workloads as W
from stardust_amd.scene import SphereScene

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module", autouse=True)
def gpu():
    L.require_gpu()


# 262,144 spheres: the limit is 1,024; 600,003: 2,343; 1,100,000: 4,296. The
# speeds put the changes below and above it; with shear a band of spheres
# crosses one cell boundary together, so that its keys fall into few blocks.
@pytest.mark.parametrize("n,speed,shear", [(262144, 10.0, False), (600003, 10.0, False), (600003, 50.0, False),
                                           (1100000, 10.0, False), (600003, 2.0, True)])
def test_large_resort(oracle, n, speed, shear):
    print("[gpu-case] large re-sort", n, speed, shear, flush=True)
    rng = np.random.default_rng(n + int(speed))
    cell, m = 0.02, int(np.ceil(n ** (1 / 3)))
    i = rng.permutation(m ** 3)[:n]
    p = ((np.stack([i % m, (i // m) % m, i // (m * m)], 1) + rng.uniform(0.0, 1.0, (n, 3))) * cell).astype(np.float32)
    r = rng.uniform(0.0005, 0.0015, n).astype(np.float32)
    v = rng.normal(0, speed, (n, 3)).astype(np.float32)
    if shear:
        band = np.abs(p[:, 2] - 10 * cell) < 0.1 * cell
        v[band, 2] = np.where(p[band, 2] < 10 * cell, 1, -1) * 200.0
    hi = (m * cell,) * 3
    g = W.grid_for((0, 0, 0), hi, cell)
    law = L.ContactParams.make(1e3, 0.3, 0.5, 2e-6, walls=((0, 0, 0), hi), max_contacts=16)
    mass = W.sphere_mass(r)
    cols = [np.ascontiguousarray(a) for a in (p[:, 0], p[:, 1], p[:, 2], v[:, 0], v[:, 1], v[:, 2])]
    sc = SphereScene(g, law, key64=True)
    sc.upload(*cols[:3], r, mass, vx=cols[3], vy=cols[4], vz=cols[5])
    st = oracle.SphereState(*cols[:3], r, mass, vx=cols[3], vy=cols[4], vz=cols[5], max_contacts=16)
    counts = []
    for k in (1, 2, 5):
        sc.step(k)
        st.step(g, law, nsteps=k, nthreads=8)
        counts.append(sc.cell_changes())
    got, exp = sc.download(), st.by_id()
    for k, (arr, col) in {"x": ("pos4", 0), "y": ("pos4", 1), "z": ("pos4", 2), "vx": ("vel4", 0), "vz": ("vel4", 2),
                          "wx": ("omg4", 0), "wy": ("omg4", 1)}.items():
        assert np.array_equal(got[k], exp[arr][:, col]), k
    limit = max(1024, n // 256)
    print("[gpu-case] changes", counts, "limit", limit, flush=True)
    assert all(full == (c > limit) for c, full in counts)
    assert max(c for c, _ in counts) > 500  # (the band of the shear case has crossed after a few steps)
    sc.close()


@pytest.mark.parametrize("speed", [3.0, 150.0])
def test_cell_changes_of_either_key_width(speed):
    """Contexts of 32-bit and of 64-bit keys step alike and report the same changes."""
    print("[gpu-case] cell changes by key width", speed, flush=True)
    rng = np.random.default_rng(17)
    n, cell, m = 20000, 0.02, 28
    p = (rng.uniform(0.02, m - 0.02, (n, 3)) * cell).astype(np.float32)
    r = rng.uniform(0.0005, 0.0015, n).astype(np.float32)
    v = rng.normal(0, speed, (n, 3)).astype(np.float32)
    hi = (m * cell,) * 3
    cols = [np.ascontiguousarray(a) for a in (*p.T, *v.T)]
    law = L.ContactParams.make(1e3, 0.3, 0.5, 1e-5, walls=((0, 0, 0), hi), max_contacts=16)
    got = []
    for key64 in (False, True):
        sc = SphereScene(W.grid_for((0, 0, 0), hi, cell), law, key64=key64)
        sc.upload(*cols[:3], r, W.sphere_mass(r), vx=cols[3], vy=cols[4], vz=cols[5])
        seen = [sc.cell_changes()]
        for k in (1, 2, 7):
            sc.step(k)
            seen.append(sc.cell_changes())
        sc.load(sc.save())
        seen.append(sc.cell_changes())
        got.append(seen)
        sc.close()
    assert got[0] == got[1]
    assert got[0][0] == got[0][-1] == (0, True)
    assert all(c > 0 and full == (c > 1024) for c, full in got[0][1:-1])
    assert got[0][-2][1] == (speed > 100.0)
