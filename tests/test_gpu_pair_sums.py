"""The pair sums (pair_region) and the corner peak's group sums (group_sums)
against the oracle at the kernel's own points, where they can go wrong: widths
from 1 down past 2^-13 and widths that are no power of two, the Gaussian's cosh
table at its ends and past it, lists that end inside a tile, and regions out of
the sums' range among regions within it.

Each flat list runs through eval_genz and as a loop's launch does
(pagani_genz_eval_launch, _launch below), which takes the pair sums without
tables. The level-form lists run the kernel with the tables: past their last
level, past the cosh rows in LDS, and with an end
inside a tile and a workgroup, bit for bit with the launches without tables.

Tolerances are test_gpu_eval's: 1e-13 of each region's scale plus the FP64
floor of f at those points, and the error and split-axis rules given there.
"""
import ctypes

import numpy as np
import pytest

import oracle_api as O
from test_gpu_eval import check_region_parity, genz_params, gpu_eval, to_dev

pytestmark = pytest.mark.gpu

pg = pytest.importorskip("gpuintegration_amd")


class _Args(ctypes.Structure):  # pagani_eval_args
    _fields_ = ([("n", ctypes.c_size_t)]
                + [(k, ctypes.c_void_p) for k in ("L", "H", "est", "err", "dim", "stream")]
                + [("consts", pg.EvalConsts)]
                + [(k, ctypes.c_void_p) for k in ("dev", "L2", "H2", "pdim", "pdim2", "fevals")])


def _launch(gpu, family, a, u, L, H, h0=None):
    """(est, err, dim) of one launch, one wave per batch: H holds widths, or with h0 the levels of widths
    h0 2^-level."""
    import torch
    d, n = L.shape
    Ld = to_dev(np.ascontiguousarray(L.ravel()), gpu)
    Hd = torch.from_numpy(np.ascontiguousarray(H.ravel())).to(gpu)
    est = torch.empty(n, dtype=torch.float64, device=gpu)
    err, dim = torch.empty_like(est), torch.empty(n, dtype=torch.uint8, device=gpu)
    with pg.Workspace(d, 0) as ws:
        ws.set_slices(1)
        args = _Args(n=n, L=Ld.data_ptr(), H=Hd.data_ptr(), est=est.data_ptr(), err=err.data_ptr(),
                     dim=dim.data_ptr())
        rc = ws.lib.pagani_ws_eval_consts(ws._ws, None, None, n, ctypes.byref(args.consts))
        assert (rc, args.consts.ndim, args.consts.slices) == (0, d, 1)
        if h0 is not None:
            assert Hd.dtype == torch.int16
            args.consts.levels = 1
            args.consts.h0[:d] = [h0] * d
        torch.cuda.synchronize()
        g = pg.genz(family, a, u)
        assert ws.lib.pagani_genz_eval_launch(ctypes.byref(g), 64, ctypes.byref(args)) == 0
        torch.cuda.synchronize()
    return est.cpu().numpy(), err.cpu().numpy(), dim.cpu().numpy().astype(np.int32)


def _compare(pg, gpu, family, a, u, L, H, slices=1):
    d, n = L.shape
    if slices == 1 and family != "corner_peak":
        got = _launch(gpu, family, a, u, L, H)
        Lr, Hr = np.ascontiguousarray(L.ravel()), np.ascontiguousarray(H.ravel())
        want = O.eval_regions_kform(d, family, O.params(a, u), Lr, Hr, n)
        check_region_parity(d, family, *got, *want, floor=True)
    L, H = np.ascontiguousarray(L.ravel()), np.ascontiguousarray(H.ravel())
    with pg.Workspace(d, 0) as ws:
        ws.set_slices(slices)
        ge, gerr, gdim = gpu_eval(ws, gpu, family, a, u, L, H, n)
    oe, oerr, odim, fd, rs = O.eval_regions_kform(d, family, O.params(a, u), L, H, n)
    check_region_parity(d, family, ge, gerr, gdim, oe, oerr, odim, fd, rs, floor=True)


def _boxes(rng, H):
    return np.floor(rng.random(H.shape) / H) * H


@pytest.mark.parametrize("family", ["gaussian", "c0", "discontinuous", "product_peak"])
@pytest.mark.parametrize("d,n", [(2, 1), (2, 64 * 8 + 1), (3, 255), (5, 321), (8, 700), (10, 130)])
@pytest.mark.parametrize("third", [False, True])
def test_widths_in_and_out_of_the_tables(pg, gpu, family, d, n, third):
    rng = np.random.default_rng(1000 * d + n)
    a, u = genz_params(family, d, seed=17 + d)
    H = 0.5 ** rng.integers(0, 14 if d < 5 else 16, size=(d, n))
    if third:
        H = np.where(rng.random((d, n)) < 0.5, H / 3, H)
    _compare(pg, gpu, family, a, u, _boxes(rng, H), H)


@pytest.mark.parametrize("d", [2, 8])
def test_gaussian_at_the_ends_of_its_table(pg, gpu, d):
    # y = 2 a^2 (c - u) h from 0 past the table's 100, the centre's sum
    # within the factored range on most regions
    n = 640
    rng = np.random.default_rng(d)
    a, u = [25.0] + [4.0] * (d - 1), [0.5] * d
    H = np.full((d, n), 0.125)
    H[0] = np.linspace(0.01, 0.9, n)
    L = rng.random((d, n)) * (1.0 - H)
    y = 2 * a[0] ** 2 * np.abs(L[0] + H[0] / 2 - u[0]) * H[0]
    assert (y > 100).any() and (y < 100).any() and ((y > 99) & (y < 101)).any()
    _compare(pg, gpu, "gaussian", a, u, L, H)


@pytest.mark.parametrize("d", [2, 3, 10])
@pytest.mark.parametrize("first", [1e8, 4e13, 1e16])
def test_product_peak_at_the_end_of_its_range(pg, gpu, d, first):
    # v = a (x - u) up to 1e13 is within the pair sums' range; 4e13 has regions on both sides
    n = 64 * 5 + 3
    rng = np.random.default_rng(d)
    a, u = [first] + [9.0] * (d - 1), [0.4] * d
    H = 0.5 ** rng.integers(1, 9, size=(d, n))
    _compare(pg, gpu, "product_peak", a, u, _boxes(rng, H), H)


@pytest.mark.parametrize("d", [2, 3, 5, 8])
@pytest.mark.parametrize("slices", [1, 2, 4, 8])
@pytest.mark.parametrize("first", [9.0, 1e31])
def test_corner_peak_groups(pg, gpu, d, slices, first):
    # a base past 1e30 leaves the groups' range: with the large coefficient
    # only the boxes at the origin stay within it, in one wave with the others
    n = 64 * 3 + 5
    rng = np.random.default_rng(10 * d + slices)
    a = [first] + [0.05] * (d - 1)
    H = 0.5 ** rng.integers(1, 7, size=(d, n))
    L = _boxes(rng, H)
    L[0, ::3] = 0.0
    _compare(pg, gpu, "corner_peak", a, [0.0] * d, L, H, slices)


def _fma(x, y, z):
    return (x.astype(np.longdouble) * y + z).astype(np.float64)


def _point_by_point(pg, family, a, u, L, H):
    """The rule's estimates of regions, every point of it by itself: in extended precision, in FP64 with the
    kernel's centred points, and the sum of the terms' magnitudes."""
    d, n = L.shape
    k2 = 1.0  # the product peak's constant, as the descriptor's integrand holds it
    for v in a:
        k2 *= v * v
    w, _, _, _, sb, _ = pg.rule_tables(d)
    set_of = np.repeat(np.arange(9), np.diff(sb))
    a, u = np.array(a)[:, None], np.array(u)[:, None]
    x0, ld = (L + H / 2 - u if family == "product_peak" else L + H / 2) * a, np.longdouble
    exact, scale, sums = np.zeros(n, ld), np.zeros(n, ld), np.zeros((9, n))
    for p, s in enumerate(set_of):
        g = np.array([pg.rule_point(d, p, j) for j in range(d)])[:, None]
        x = (L.astype(ld) + H.astype(ld) / 2) - g.astype(ld) * H
        v = _fma(-g, H * a, x0)
        if family == "corner_peak":
            fx = (1 + (a * x).sum(0)) ** -(d + 1)
            b = np.ones(n)
            for j in range(d):
                b = b + v[j]
            f, q = np.ones(n), b
            for j in range(d):
                q = q * b
            f = 1.0 / q
        else:
            fx = ld(k2) / (1 + (a.astype(ld) * (x - u)) ** 2).prod(0)
            q = np.ones(n)
            for j in range(d):
                q = q * _fma(v[j], v[j], 1.0)
            f = k2 / q
        exact += ld(w[s][0]) * fx
        scale += abs(ld(w[s][0])) * fx
        sums[s] += f
    plain = np.zeros(n)
    for s in range(9):
        plain = _fma(np.full(n, w[s][0]), sums[s], plain)
    return exact, plain, scale


@pytest.mark.parametrize("family", ["corner_peak", "product_peak"])
@pytest.mark.parametrize("d", [2, 3, 5])
def test_rounding_is_that_of_single_points(pg, gpu, family, d):
    """Sums over groups of points round no worse than the points one by one: the root mean square of the
    regions' errors against extended precision, within 1.25 (a group's last roundings are shared by its
    points, those of single points average out)."""
    n = 20000 if d < 5 else 6000
    rng = np.random.default_rng(40 + d)
    a, u = genz_params(family, d, seed=3)
    H = 0.5 ** rng.integers(1, 7, size=(d, n))
    L = _boxes(rng, H)
    exact, plain, scale = _point_by_point(pg, family, a, u, L, H)
    rms = lambda est: float(np.sqrt((((est - exact) / scale) ** 2).mean()))  # noqa: E731
    vol = H.prod(0)  # a power of two
    with pg.Workspace(d, 0) as ws:
        for slices in ((1, 4) if family == "corner_peak" else (1,)):
            ws.set_slices(slices)
            est = gpu_eval(ws, gpu, family, a, u, np.ascontiguousarray(L.ravel()),
                           np.ascontiguousarray(H.ravel()), n)[0]
            assert rms(est / vol) <= 1.25 * rms(plain)


# n = 262144 regions is the first list the kernel with tables takes; eight waves a workgroup, four with a mask
@pytest.mark.parametrize("family", ["gaussian", "c0", "discontinuous"])
@pytest.mark.parametrize("d,n", [(2, 262144), (2, 262144 + 64 * 5 + 1), (3, 262144 + 64 * 9 + 33),
                                 (8, 262144 + 64 * 3 + 63)])
@pytest.mark.parametrize("h0", [1.0, 1.0 / 3.0])
def test_tables(pg, gpu, family, d, n, h0):
    """A long level-form list, as doubles and in short lists the same bits; and the oracle's on a sample."""
    rng = np.random.default_rng(7 * d + n)
    a, u = genz_params(family, d, seed=23 + d)
    if family == "gaussian":  # rows past the LDS part of the cosh table, and past the table
        a[0] = 40.0
    last = max(96 // d, 12)  # levels with a table entry: 0 .. last - 1
    lev = rng.integers(0, last + 3, size=(d, n)).astype(np.int16)
    lev[:, ::2] = rng.integers(0, 5, size=(d, (n + 1) // 2))
    H = np.ldexp(h0, -lev.astype(np.int32))
    L = np.floor(rng.random((d, n)) * (1.0 - H) / H) * H
    assert (lev == 0).any() and (lev == last - 1).any() and (lev >= last).any()
    if family == "gaussian":
        row = 2 * np.abs(2 * a[0] ** 2 * (L[0] + H[0] / 2 - u[0]) * H[0])
        assert (row < 51).any() and ((row > 51) & (row < 200)).any() and (row > 201).any()
    long = _launch(gpu, family, a, u, L, lev, h0)
    for part in (slice(0, 200001), slice(200001, n)):
        for got in (_launch(gpu, family, a, u, L[:, part], lev[:, part], h0),
                    _launch(gpu, family, a, u, L[:, part], H[:, part])):
            for x, y in zip(long, got):
                assert np.array_equal(x[part], y)
    pick = np.concatenate([np.arange(300), n - 1 - np.arange(300)])
    pick = pick[(lev[:, pick] < 12).all(0)]
    assert pick.size > 100
    Lp, Hp = (np.ascontiguousarray(x[:, pick].ravel()) for x in (L, H))
    want = O.eval_regions_kform(d, family, O.params(a, u), Lp, Hp, pick.size)
    check_region_parity(d, family, *(x[pick] for x in long), *want, floor=True)
