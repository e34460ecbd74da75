"""The sweep over one scene with its candidates taken from bitmaps, against the
oracle's sweep that tests every candidate, pair for pair in order: slices that
are full, end early or hold one box; boxes in few bins, in all of them, far from
the others; equal and touching boxes; zeros of both signs, infinite, inverted and
undefined bounds."""
import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import hulls as H

pytestmark = pytest.mark.gpu


def boxes(n, case, rng):
    lo, hi = np.zeros((n, 4), np.float32), np.zeros((n, 4), np.float32)
    c = rng.uniform(0, 1, (n, 3)).astype(np.float32)
    r = (rng.uniform(0.2, 1, (n, 3)) * 0.6 * n ** (-1 / 3)).astype(np.float32)
    if case == "equal":
        c[:], r[:] = 0.5, 0.25
    elif case == "touching":  # faces on a lattice
        c, r = np.round(c * 16).astype(np.float32), np.full((n, 3), 0.5, np.float32)
    elif case == "flat":
        c[:, 1] = 0.25
        r[:, 1] = 0.0
    elif case == "large":
        r[::7] *= 20
    elif case == "far":
        c[::50] += rng.choice([-1e6, 1e6, 1e30], (len(c[::50]), 3)).astype(np.float32)
    elif case == "zeros":
        c = np.round(c * 4 - 2).astype(np.float32) * np.float32(-0.0) + np.round(c * 2 - 1).astype(np.float32)
        r[:] = 0.0
    lo[:, :3], hi[:, :3] = c - r, c + r
    if case == "odd":
        k = np.arange(0, n, 5)
        lo[k[0::5], rng.integers(0, 3)] = -np.inf
        hi[k[1::5], rng.integers(0, 3)] = np.inf
        lo[k[2::5], 1], hi[k[2::5], 1] = hi[k[2::5], 1], lo[k[2::5], 1]  # inverted
        lo[k[3::5], :3], hi[k[3::5], :3] = hi[k[3::5], :3], lo[k[3::5], :3]
        lo[k[4::5], :3] = hi[k[4::5], :3] = np.inf
    elif case == "undefined":
        m = rng.uniform(0, 1, (n, 3)) < 0.05
        lo[:, :3][m] = np.nan
        hi[:, :3][rng.uniform(0, 1, (n, 3)) < 0.03] = np.nan
        lo[::11, :3] = np.float32(-np.nan)
    return lo, hi


@pytest.mark.parametrize("case,n", [("random", 1), ("random", 2), ("random", 255), ("random", 256), ("random", 257),
                                    ("random", 3000), ("random", 20000), ("equal", 300), ("touching", 4000),
                                    ("flat", 2000), ("large", 2000), ("far", 3000), ("zeros", 700), ("odd", 1500),
                                    ("undefined", 1500)])
def test_pairs_in_order(oracle, case, n):
    print("[gpu-case] sap bins", case, n, flush=True)
    L.require_gpu()
    lo, hi = boxes(n, case, np.random.default_rng(n))
    d = H.DeviceHulls(H.generate_hulls(0x5EEDC400, n))
    d.lo4.upload(lo)
    d.hi4.upload(hi)
    most = n * (n - 1) // 2 + 16
    pairs, npairs, axis = d.sap(capacity=min(most, 4_000_000))
    got = pairs.download(np.int32, 2 * npairs).reshape(-1, 2)
    want, _ = oracle.sap_pairs(lo, hi, axis=axis)
    assert np.array_equal(got, want)
