"""The rules by which the host plans steps on lists (sd_list_plan.hpp), run
against a simulated device: bodies that move by so much a step, at such a
distance from the origin, whose lists are built, used up and given up as the
kernels do. What is counted is what a caller pays for: steps that build, steps
queued that a given-up sequence drops, launch sequences."""
import ctypes as C
import os
import subprocess

import numpy as np
import pytest

CSRC = os.path.join(os.path.dirname(os.path.dirname(os.path.abspath(__file__))), "stardust_amd", "csrc")
SRC = r"""
#include "sd_list_plan.hpp"
using namespace sd;
struct Run { long long steps, built, on_lists, dropped, sequences; };
// move[i]: movement of step i; far: largest coordinate; over: the lists are too short; call: steps of a call
extern "C" Run simulate(const float* move, int n, float size, float far, int over, int call) {
    Run r = {};
    ListPlan plan;
    float displaced = 0.0f, margin = 0.0f, limit = 0.0f, last = 0.0f;
    for (int at = 0; at < n;) {
        const float largest = clump_largest(size);
        const ListRun q = plan.next(std::min(n, (at / call + 1) * call) - at, plan.pays(largest), false, largest,
                                    CL_MARGIN_KEPT * clump_margin(plan.last, size));
        const int first = at;
        bool given_up = false;
        for (int k = 0; k < q.none; ++k) last = at ? move[at - 1] : 0.0f, ++at;
        for (int k = 0; k < q.build + q.use; ++k) {
            const float m = at ? move[at - 1] : 0.0f;
            if (k < q.build) {
                margin = clump_build_margin(m, size, far);
                limit = clump_limit(margin, far);
                displaced = 0.0f;
                r.built += 1;
            } else if (!(displaced + m <= limit) || over) {
                given_up = true;
                r.dropped += q.build + q.use - k;
                break;
            } else {
                displaced += m;
                r.on_lists += 1;
            }
            last = m;
            ++at;
        }
        if (at == first && !given_up) { r.steps = -1; return r; }  // no progress
        ListReport p;
        p.ran = at - first;
        p.given_up = given_up;
        p.crowded = over && q.none == 0;
        p.last = last;
        p.budget = limit;
        p.used = displaced;
        p.lost = CL_MARGIN_KEPT * margin - limit;
        plan.read(p, q.none == 0, largest);
        r.sequences += 1;
    }
    r.steps = n;
    return r;
}
"""


class Run(C.Structure):
    _fields_ = [(k, C.c_longlong) for k in ("steps", "built", "on_lists", "dropped", "sequences")]


@pytest.fixture(scope="module")
def lib(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "plan.cpp").write_text(SRC)
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-fPIC", "-shared", "-I", CSRC,
                    str(d / "plan.cpp"), "-o", str(d / "libplan.so")], check=True)
    x = C.CDLL(str(d / "libplan.so"))
    x.simulate.restype = Run
    x.simulate.argtypes = [C.c_void_p, C.c_int, C.c_float, C.c_float, C.c_int, C.c_int]
    return x


def simulate(lib, move, size, far, over=0, call=1 << 20):
    move = np.ascontiguousarray(move, np.float32)
    r = lib.simulate(move.ctypes.data, len(move), size, far, over, call)
    assert r.steps == len(move)
    return r


N, SIZE = 4000, 0.02


# bodies of 2 cm at rest, slow, and moving as far as lists pay for, near the
# origin and as far from it as the widest margin covers
@pytest.mark.parametrize("far", [0.1, 30.0, 300.0, 1500.0])
@pytest.mark.parametrize("move", [0.0, 1e-9, 1e-7, 2e-6])
def test_lists_last(lib, move, far):
    r = simulate(lib, np.full(N, move), SIZE, far)
    assert r.on_lists > 0.9 * N and r.dropped <= 2 * 64, [getattr(r, k) for k, _ in Run._fields_]


# beyond: lists are tried once in a while only, and little is queued for nothing
@pytest.mark.parametrize("far", [2100.0, 1e4, 1e6])
@pytest.mark.parametrize("move", [0.0, 1e-7, 1e-4])
def test_lists_rest_far_from_the_origin(lib, move, far):
    r = simulate(lib, np.full(N, move), SIZE, far)
    assert r.built <= N / 200 and r.dropped <= 3 * r.built and r.sequences < N / 25, \
        [getattr(r, k) for k, _ in Run._fields_]


# the most that rounding leaves is used up in a few steps: at any distance the
# sequences that drop steps are few
@pytest.mark.parametrize("far", [0.1, 500.0, 1000.0, 1500.0, 1900.0, 1990.0])
def test_few_steps_dropped_at_any_speed(lib, far):
    for move in np.geomspace(1e-8, 1e-3, 60):
        r = simulate(lib, np.full(N, move), SIZE, far)
        assert r.dropped <= max(8, 0.05 * N), (move, [getattr(r, k) for k, _ in Run._fields_])


def test_speeds_that_change(lib):
    """Spikes, and a slow growth: lists come back after each, most steps use them."""
    spikes = np.full(N, 1e-6)
    spikes[::500] = 1e-2
    growth = np.geomspace(1e-8, 1e-5, N)
    for move in (spikes, growth):
        r = simulate(lib, move, SIZE, 1.0)
        assert r.on_lists > 0.7 * N, [getattr(r, k) for k, _ in Run._fields_]


# calls of many steps, of a few, and of one (as a profile makes them)
@pytest.mark.parametrize("call", [1 << 20, 10, 1])
def test_lists_too_short_rest(lib, call):
    r = simulate(lib, np.full(N, 1e-6), SIZE, 1.0, over=1, call=call)
    assert r.built <= N / 100 and r.dropped <= 3 * r.built


@pytest.mark.parametrize("call", [10, 1])
def test_calls_of_few_steps(lib, call):
    r = simulate(lib, np.full(N, 1e-6), SIZE, 1.0, call=call)
    assert r.on_lists > 0.9 * N and r.dropped <= 2 * 64
