"""State read-back against the saved state: the rows in slot order and the ids
of sd_ctx_save hold the same values (exact)."""
import struct
import sys

import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import workloads as W
from stardust_amd.scene import SphereScene

pytestmark = pytest.mark.gpu
NAMES = ("x", "y", "z", "vx", "vy", "vz", "wx", "wy", "wz")


@pytest.fixture(scope="module", autouse=True)
def gpu():
    L.require_gpu()


def scene(n, key64):
    """Spheres on a jittered lattice in fast motion: the slot order differs from the id order."""
    rng = np.random.default_rng(n)
    m = int(np.ceil(n ** (1 / 3)))
    i = rng.permutation(m ** 3)[:n]
    p = (np.stack([i % m, (i // m) % m, i // (m * m)], 1) + 0.5 + rng.uniform(-0.1, 0.1, (n, 3))) * 0.02
    r = rng.uniform(0.004, 0.008, n).astype(np.float32)
    v = rng.normal(0, 1.0, (n, 3)).astype(np.float32)
    hi = (m * 0.02,) * 3
    sc = SphereScene(W.grid_for((0, 0, 0), hi, 0.02),
                     L.ContactParams.make(1e5, 0.3, 0.5, 1e-5, walls=((0, 0, 0), hi), max_contacts=8), key64=key64)
    p = p.astype(np.float32)
    sc.upload(p[:, 0], p[:, 1], p[:, 2], r, W.sphere_mass(r), vx=v[:, 0], vy=v[:, 1], vz=v[:, 2])
    return sc


def saved(sc):
    """Rows by id from the saved state: header (48 bytes), pos4, vel4, omg4, ids."""
    buf, n = sc.save(), sc.n
    head = struct.calcsize("<IIiiiiqiiQ")
    rows = buf[head:head + 48 * n].view(np.float32).reshape(3, n, 4)
    ids = buf[head + 48 * n:head + 52 * n].view(np.int32)
    out = np.empty((3, n, 4), np.float32)
    out[:, ids] = rows
    return {k: out[j // 3, :, j % 3] for j, k in enumerate(NAMES)}


# one chunk, exactly one, one more, several chunks per thread with a remainder
@pytest.mark.parametrize("n", [1, 257, 32768, 32769, 500003])
@pytest.mark.parametrize("key64", [False, True])
def test_sphere_readback(n, key64):
    print("[gpu-case] sphere read-back", n, key64, flush=True)
    sys.stdout.flush()
    sc = scene(n, key64)
    sc.step(3)
    exp = saved(sc)
    got = sc.download()
    for k in NAMES:
        assert np.array_equal(got[k], exp[k]), k
    # a part of the arrays only; the state is untouched by a read-back
    part = {k: np.full(n, np.nan, np.float32) for k in ("y", "vx", "wz")}
    L.call("sd_ctx_download_spheres", sc.h, *[L.ptr(part[k]) if k in part else None for k in NAMES])
    for k, v in part.items():
        assert np.array_equal(v, exp[k]), k
    L.call("sd_ctx_download_spheres", sc.h, *[None] * 9)
    sc.step(2)
    exp, got = saved(sc), sc.download()
    for k in NAMES:
        assert np.array_equal(got[k], exp[k]), k
    sc.close()
