"""Neighbour pairs whose partners are kept between the count and the output,
against the oracle's search: spheres with fewer partners than are kept, as many
and more (searched again), scratch that holds all, some or none of them, one cell
and cells at the grid's edges, sizes around a block."""
import ctypes as C

import numpy as np
import pytest

from stardust_amd import _lib as L

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n,cells,r", [(1, 1, 0.4), (2, 1, 0.4), (9, 1, 0.9), (10, 1, 0.9), (40, 1, 0.9), (127, 4, 0.4),
                                       (128, 4, 0.5), (129, 5, 0.5), (1000, 7, 0.3), (1000, 7, 0.6), (5000, 11, 0.5),
                                       (3000, 40, 0.5)])
@pytest.mark.parametrize("kept", [8, 3, 0])
def test_pairs(oracle, n, cells, r, kept):
    print("[gpu-case] neighbour pairs", n, cells, r, kept, flush=True)
    L.require_gpu()
    rng = np.random.default_rng(n + cells)
    pos = np.zeros((n, 4), np.float32)
    pos[:, :3] = rng.uniform(-0.2, cells + 0.2, (n, 3))  # some outside: the cells at the edges take them
    pos[:, 3] = rng.uniform(0.2 * r, r, n)
    g = L.Grid.make((0.0, 0.0, 0.0), 1.0, [cells, cells + 1, max(cells - 1, 1)])
    keys, _ = oracle.hash_keys(*[np.ascontiguousarray(a) for a in pos[:, :3].T], g)
    order = np.argsort(keys, kind="stable")
    pos = np.ascontiguousarray(pos[order])
    ranges = oracle.cell_ranges_u32(np.ascontiguousarray(keys[order]), g.n_cells)
    want = oracle.neighbor_pairs(pos, g, ranges, 0.05)
    nb = C.c_size_t()
    L.call("sd_neighbor_pairs_scratch_bytes", n, C.byref(nb))
    size = nb.value - 4 * n * (8 - kept)
    p4, rg, scratch = L.DeviceBuffer.from_array(pos), L.DeviceBuffer.from_array(ranges), L.DeviceBuffer(size)
    cap = len(want) + 3
    out = L.DeviceBuffer(8 * cap)
    got = C.c_int()
    call = lambda capacity, bytes_: L.load().sd_neighbor_pairs(p4.ptr, n, C.byref(g), rg.ptr, 0.05, out.ptr, capacity,
                                                               C.byref(got), scratch.ptr, bytes_, None)
    assert call(cap, size) == L.SD_OK and got.value == len(want)
    assert np.array_equal(out.download(np.int32, 2 * got.value).reshape(-1, 2), want)
    if len(want) > 2:
        half = len(want) // 2
        assert call(half, size) == L.SD_ERR_CAPACITY and got.value == len(want)
        assert np.array_equal(out.download(np.int32, 2 * half).reshape(-1, 2), want[:half])
    assert call(cap, nb.value - 32 * n - 1) == L.SD_ERR_ARG
