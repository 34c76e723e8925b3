"""Error estimates that a change of rounding moves.

The null rules of a smooth integrand cancel to 1e-8 .. 1e-11 of their terms,
and an FP32 integrand's to the rounding of its values, so one more or one less
contraction anywhere in an evaluation changes the errors a caller sees in
their fifth digit or before.  Each route of these integrands has one order of
operations, and the values are that order's, bit for bit.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

DIMS = (2, 3, 4, 5, 6, 8, 10)


def _params(fam, d):
    rng = np.random.default_rng(100 * d + len(fam))
    lo, hi = {"oscillatory": (1.0, 1.5), "gaussian": (9.0, 11.0)}.get(fam, (5.0, 15.0))
    return rng.uniform(lo, hi, d).tolist(), rng.uniform(0.3, 0.7, d).tolist()


def segments(pg, d):
    """errorest of an oscillatory integral run whole in the segment kernel"""
    b = pg.Batch(0, workers=1)
    b.set_segments(65536)
    items = [("oscillatory", *_params("oscillatory", d), eps) for eps in (1e-2, 1e-6)]
    results, codes = b.integrate(items)
    assert codes == [0, 0] and b.stats()["segment_integrals"] == 2
    b.close()
    return [r.errorest.hex() for r in results]


SEGMENTS = {
    2: ["0x1.021d46fa4d5b8p-40", "0x1.021d46fa4d5b8p-40"],
    3: ["0x1.a1770e5958866p-37", "0x1.a1770e5958866p-37"],
    4: ["0x1.0d5866bd20f20p-35", "0x1.0d5866bd20f20p-35"],
    5: ["0x1.7e58e05fb80fap-31", "0x1.7e58e05fb80fap-31"],
    6: ["0x1.5599b5dc1981fp-27", "0x1.5599b5dc1981fp-27"],
    8: ["0x1.feadc98cffedep-26", "0x1.feadc98cffedep-26"],
    10: ["0x1.23458138c747dp-24", "0x1.23458138c747dp-24"],
}


@pytest.mark.parametrize("d", DIMS)
def test_oscillatory_segments(pg, gpu, d):
    assert segments(pg, d) == SEGMENTS[d]
