"""How a Krylov solve hands its iterations to the device (csrc/solve_plan.h,
host arithmetic): a solve as long as the last one is looked at once, and one
much longer than it is neither stopped at every iteration nor launched far past
its end."""
import ctypes as C
import math
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
SRC = """
#include "solve_plan.h"
extern "C" int batch(int pred, int maxit, int launched) { return sph::SolvePlan{pred, maxit}.batch(launched); }
extern "C" int run_graph(int pred, int maxit, int launched, int left) {
    return sph::SolvePlan{pred, maxit}.run_graph(launched, left) ? sph::KR_RUN : 1;
}
"""


@pytest.fixture(scope="module")
def plan(tmp_path_factory):
    d = tmp_path_factory.mktemp("plan")
    (d / "p.cpp").write_text(SRC)
    so = str(d / "p.so")
    subprocess.check_call(["g++", "-std=c++17", "-shared", "-fPIC", "-I",
                           os.path.join(ROOT, "urban-sph_a100_amd", "csrc"), str(d / "p.cpp"), "-o", so])
    return C.CDLL(so)


def _solve(plan, pred, need, maxit=5000):
    """looks, iterations launched, graphs launched of a solve of `need` iterations."""
    looks = launched = graphs = 0
    first = pred > 0
    while (first or launched < need) and launched < maxit:
        n = plan.batch(pred, maxit, launched)
        assert 1 <= n <= maxit - launched
        b = 0
        while b < n:
            b += plan.run_graph(pred, maxit, launched, n - b)
            graphs += 1
        assert b == n
        launched += n
        looks += 1
        first = False
    return looks, launched, graphs


@pytest.mark.parametrize("pred", [1, 3, 8, 9, 40, 300])
def test_as_predicted(plan, pred):
    looks, launched, _ = _solve(plan, pred, pred)
    assert launched <= pred + 2
    assert looks == 1 if pred <= 8 else looks <= 2 + (pred - pred * 9 // 10 + 5) // 2


@pytest.mark.parametrize("pred,need", [(p, n) for p in (1, 4, 8, 9, 20) for n in (10, 44, 150, 400, 3000) if n > p])
def test_much_longer_than_predicted(plan, pred, need):
    """Looks and iterations past the end both grow with the root of the excess;
    one look an iteration would be its half or more."""
    looks, launched, graphs = _solve(plan, pred, need)
    excess = need - pred
    assert looks <= 6 + 1.5 * math.sqrt(2 * excess)
    assert launched - need <= max(2, math.sqrt(2 * (launched - pred)))
    if excess >= 400:
        assert graphs <= 64 + launched // 2   # mostly graphs of four


@pytest.mark.parametrize("need", [1, 10, 44, 400])
def test_without_prediction(plan, need):
    looks, launched, _ = _solve(plan, 0, need)
    assert looks <= 16 and launched <= 4 + need + need // 2


def test_iteration_cap(plan):
    for pred in (0, 1, 8, 50):
        for maxit in (1, 2, 7, 33):
            assert _solve(plan, pred, 10 ** 6, maxit)[1] == maxit
