"""The iteration loop of short lists in one workgroup against the host-driven
loop: every value is formed in the same order, so results, traces and region
counts agree bit for bit -- at every slice count, with widths as levels and as
doubles, on lists of less than a wave, of one chunk and of two, across the
hand-over to the launches, with a list of the caller's, and where the host
finishes an iteration (a small memory model)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

FAMILIES = ("oscillatory", "product_peak", "corner_peak", "gaussian", "c0", "discontinuous")


def _params(fam, d, seed):
    rng = np.random.default_rng(seed)
    lo, hi = {"oscillatory": (1.0, 1.5), "gaussian": (9.0, 11.0)}.get(fam, (5.0, 15.0))
    return rng.uniform(lo, hi, d).tolist(), rng.uniform(0.3, 0.7, d).tolist()


def _both(pg, fam, d, eps, setup=lambda ws: None, **kw):
    a, u = _params(fam, d, d * 31 + len(fam))
    got = []
    for device in (False, True):
        with pg.Workspace(d, 0) as ws:
            ws.set_device_loop(device)
            setup(ws)
            r = ws.integrate_genz(fam, a, u, epsrel=eps, epsabs=1e-20, **kw)
            tr, st = ws.trace(), ws.stats()
            got.append(((r.estimate, r.errorest, r.nregions, r.iters, r.status),
                        [list(tr[k]) for k in ("n", "m", "estimate", "errorest")],
                        st["regions_evaluated"], st))
    assert got[0][:3] == got[1][:3]
    return got[1][3]


@pytest.mark.parametrize("levels", [True, False], ids=["levels", "widths"])
@pytest.mark.parametrize("d", [2, 3, 5, 8, 10])
@pytest.mark.parametrize("fam", FAMILIES)
def test_matches_the_host_loop(pg, gpu, fam, d, levels):
    eps = {2: 1e-8, 3: 1e-6, 5: 1e-4, 8: 1e-2, 10: 1e-1}[d]
    st = _both(pg, fam, d, eps, lambda ws: ws.set_level_form(levels))
    assert st["device_rounds"] < st["device_iterations"] or st["device_iterations"] == 1
    assert st["device_iterations"] > 0


@pytest.mark.parametrize("slices", [1, 2, 4, 8])
@pytest.mark.parametrize("fam", ["oscillatory", "corner_peak", "gaussian", "c0"])
def test_slice_counts(pg, gpu, fam, slices):
    _both(pg, fam, 4, 1e-4, lambda ws: ws.set_slices(slices))


@pytest.mark.parametrize("k", [1, 2, 7, 8, 20, 26, 90])
def test_first_lists(pg, gpu, k):
    """Uniform starts of k^2 regions: one, less than a wave, ragged waves, one
    chunk, two, and more than a workgroup takes."""
    _both(pg, "gaussian", 2, 1e-7, init_k=k)
    _both(pg, "discontinuous", 2, 1e-5, init_k=k)


@pytest.mark.parametrize("mem", [200_000, 2_000_000])
def test_the_host_finishes_an_iteration(pg, gpu, mem):
    """The first list is past a tenth of the smaller model's budget (the host
    loop runs it); the larger model's run starts on the device and leaves it."""
    st = _both(pg, "gaussian", 4, 1e-6, lambda ws: ws.set_device_mem(mem))
    assert (st["device_iterations"] > 0) == (mem > 200_000)
    assert st["iterations"] > st["device_iterations"]


def test_longer_than_a_launch(pg, gpu):
    """More iterations than the first launch (24) and the first of the later
    ones (8) take, the others replayed and launched; every list within the
    workgroup's (70 tiles of a 2D discontinuous integrand)."""
    for graphs in (True, False):
        a, u = [5.0, 6.0], [0.4, 0.6]
        got = []
        for device in (False, True):
            with pg.Workspace(2, 0) as ws:
                ws.set_device_loop(device)
                ws.set_graphs(graphs)
                for _ in range(2):  # the second integral finds another one's buffers
                    r = ws.integrate_genz("discontinuous", a, u, epsrel=1e-14, epsabs=1e-300)
                got.append((r.estimate, r.errorest, r.nregions, r.iters, r.status,
                            list(ws.trace()["estimate"])))
                st, sizes = ws.stats(), ws.trace()["n"]
        assert got[0] == got[1]
        assert max(sizes) <= 70 * 64 and len(sizes) > 24 + 8
        assert st["device_iterations"] == 2 * len(sizes)
        assert st["graph_launches"] == (2 * (-(-(len(sizes) - 24) // 8) - 1) if graphs else 0)
