"""The rigid bodies' broadphase walk, whose candidates are taken four at a time,
against the oracle's steps: cells and rows that hold fewer bodies than a batch,
whole batches, and a few more; one to many scenes; grids of one cell. Exact."""
import numpy as np
import pytest

from stardust_amd import _lib as L
from stardust_amd import hullbody as HB
from test_gpu_hullbody import compare, law, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("sizes,side", [([(1, 1)], 0.03), ([(2, 1)], 0.02), ([(2, 3), (1, 4)], 0.025), ([(4, 5)], 0.03),
                                        ([(9, 8), (3, 1), (6, 7)], 0.035), ([(40, 40)], 0.06),
                                        ([(60, 9), (17, 30)], 0.05)])
def test_walk_equals_oracle(oracle, sizes, side):
    print("[gpu-case] hull walk", sizes, side, flush=True)
    L.require_gpu()
    bodies, first = HB.concat([scene(0x5B00 + 7 * k, h, s, side) for k, (h, s) in enumerate(sizes)])
    c = law()
    st = oracle.HullBodyState(bodies, first)
    sc = HB.HullBodyScene(c)
    sc.upload(bodies, first)
    for k in (1, 2, 7):
        sc.step(k)
        st.step(c, nsteps=k, nthreads=8)
        compare(sc, st, "after %d more" % k)
    sc.close()
