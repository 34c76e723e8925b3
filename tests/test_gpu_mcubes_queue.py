"""m-Cubes iterations queued without a word from the host: the estimate, the
stopping rule and the grid's refinement run on the device.  Against the oracle
at iteration counts on either side of a queue's length (16), for runs that the
stopping rule ends inside a queue, before adjusting is over and after, with
one grid for all axes; with timing on, the queue is one iteration long and the
run the same.  Tolerances are those of the whole-run comparison with the
oracle in test_gpu_mcubes.py."""
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


def test_no_iterations():
    with pg.MCubes(2) as mc:
        r = mc.integrate_genz("gaussian", [5.0, 5.0], [0.5, 0.5], epsrel=1e-3, epsabs=1e-30,
                              ncall=1e4, total_iters=0, adjust_iters=0, skip_iters=0)
        assert (r["iters"], r["status"], r["neval"]) == (0, 1, 0)
        assert np.array_equal(mc.grid(), O.mc_grid_init(2))
