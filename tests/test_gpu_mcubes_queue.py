"""m-Cubes iterations queued without a word from the host: the estimate, the
stopping rule and the grid's refinement run on the device.  Against the oracle
at iteration counts on either side of a queue's length (16), for runs that the
stopping rule ends inside a queue, before adjusting is over and after, with
one grid for all axes; with timing on, the queue is one iteration long and the
run the same.  Tolerances are those of the whole-run comparison with the
oracle in test_gpu_mcubes.py."""
import ctypes
import os

import numpy as np
import pytest

import oracle_api as O

pytestmark = pytest.mark.gpu

pg = pytest.importorskip("gpuintegration_amd")


def _check(r, trace, xi, o):
    ti, tsi = trace
    assert (r["iters"], r["status"], len(ti)) == (o["iters"], o["status"], o["iters"])
    for got, want, tol in ((ti, o["ti"], 1e-8), (tsi, o["tsi"], 1e-7)):
        want = np.asarray(want)[: len(ti)]
        assert np.max(np.abs(np.asarray(got) - want) / np.abs(want), initial=0.0) <= tol
    assert np.max(np.abs(xi - o["xi"])) <= 1e-8
    assert abs(r["estimate"] - o["estimate"]) <= 1e-8 * abs(o["estimate"])
    assert abs(r["errorest"] - o["errorest"]) <= 1e-7 * o["errorest"]


@pytest.mark.parametrize("total,adjust,skip,eps,one_axis", [
    (15, 0, 0, 1e-9, False), (16, 16, 0, 1e-9, False), (17, 1, 0, 1e-9, False),
    (33, 17, 3, 1e-9, False), (5, 12, 2, 1e-9, False), (20, 18, 16, 1e-9, True),
    (40, 20, 2, 3e-2, False), (40, 6, 2, 1.5e-3, False), (40, 3, 0, 1e-2, True)])
def test_queued_iterations_match_oracle(total, adjust, skip, eps, one_axis):
    fam, a, u = "product_peak", [6.0, 7.0, 8.0], [0.4, 0.5, 0.6]
    for timing in (False, True):
        with pg.MCubes(3) as mc:
            mc.set_timing(timing)
            r = mc.integrate_genz(fam, a, u, epsrel=eps, epsabs=1e-30, ncall=2e4,
                                  total_iters=total, adjust_iters=adjust, skip_iters=skip,
                                  one_axis=one_axis, generator="default", seed=9)
            trace, xi = mc.trace(), mc.grid()
        o = O.mc_integrate(fam, 3, O.params(a, u), eps, 1e-30, 2e4, total, adjust, skip, "default",
                           seed=9, one_axis=one_axis, trace_cap=64)
        _check(r, trace, xi, o)


@pytest.mark.parametrize("generator", ["default", "lcg"])
def test_empty_bins(generator):
    """Nine tenths of axis 0's bins and half of axis 1's hold no weight."""
    fam, a, u = "discontinuous", [5.0, 6.0], [0.1, 0.5]
    with pg.MCubes(2) as mc:
        r = mc.integrate_genz(fam, a, u, epsrel=1e-9, epsabs=1e-30, ncall=2e4, total_iters=8,
                              adjust_iters=6, skip_iters=1, generator=generator, seed=9)
        trace, xi = mc.trace(), mc.grid()
    o = O.mc_integrate(fam, 2, O.params(a, u), 1e-9, 1e-30, 2e4, 8, 6, 1, generator, seed=9,
                       trace_cap=64)
    assert np.isfinite(xi).all()
    _check(r, trace, xi, o)


def test_no_iterations():
    with pg.MCubes(2) as mc:
        r = mc.integrate_genz("gaussian", [5.0, 5.0], [0.5, 0.5], epsrel=1e-3, epsabs=1e-30,
                              ncall=1e4, total_iters=0, adjust_iters=0, skip_iters=0)
        assert (r["iters"], r["status"], r["neval"]) == (0, 1, 0)
        assert np.array_equal(mc.grid(), O.mc_grid_init(2))


def _reftests():
    return ctypes.CDLL(os.path.join(os.path.dirname(os.path.abspath(__file__)), "cxx", "libreftests.so"))


def _callback_run(eps, total, adjust, fails=0):
    first, calls, r = ctypes.c_int(), ctypes.c_int(), pg.McResult()
    rc = _reftests().reftest_mc_calls(ctypes.c_double(eps), ctypes.c_double(2e4), total, adjust, 0, fails,
                                      ctypes.byref(first), ctypes.byref(calls), ctypes.byref(r))
    assert rc == 0
    return first.value, calls.value, r


@pytest.mark.parametrize("eps,total,adjust,iters", [(1e-12, 20, 4, 20), (0.5, 40, 3, 5), (0.5, 40, 20, 5)])
def test_callback_is_called_once_per_iteration(gpu, eps, total, adjust, iters):
    """A callback need not know of iterations queued ahead: it sees the run's own, no more."""
    calls, r = _callback_run(eps, total, adjust)[1:]
    assert (r.iters, calls) == (iters, iters)


def test_a_failing_callback_leaves_the_handle_usable(gpu):
    """The run after one whose callback failed in its third iteration is the run of a fresh handle (no
    adjusting iterations: those repeat to the last bits only, their histograms being LDS additions)."""
    first, calls, r = _callback_run(1e-12, 8, 0, fails=3)
    fresh = _callback_run(1e-12, 8, 0)[2]
    assert first == pg.EUNSUPPORTED and calls == 8
    assert (r.estimate, r.errorest, r.iters, r.status) == (fresh.estimate, fresh.errorest, 8, 1)


def test_own_grid_ends_with_its_last_edge(gpu):
    """A sampling launch over a program's own grid: what lies behind the ndim x
    (PAGANI_MC_BINS + 1) edges does not decide whether it samples."""
    import torch
    edges = np.append(O.mc_grid_init(1).ravel(), 1.0)
    xi = torch.from_numpy(edges).to(gpu)
    part = (ctypes.c_double * 2)()
    rc = _reftests().reftest_mc_own_grid(ctypes.c_void_p(xi.data_ptr()), 10000, part)
    # the integral of exp(-50 (x - 0.3)^2) over [0, 1] from 2 points in each of 10^4 strata
    assert rc == 0 and abs(part[0] - 0.25032445820538396) <= 1e-4 and part[1] > 0.0
