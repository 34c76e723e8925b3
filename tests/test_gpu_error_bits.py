"""Error estimates that a change of rounding moves.

The null rules of a smooth integrand cancel to 1e-8 .. 1e-11 of their terms,
and an FP32 integrand's to the rounding of its values, so one more or one less
contraction anywhere in an evaluation changes the errors a caller sees in
their fifth digit or before.  Each route of these integrands has one order of
operations: the segment kernel, the launches at one wave per batch and at
several, the first list of less than a batch, the generic loop of FP32
integrands.  The values are that order's, bit for bit.
"""
import math

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


def short_list(pg, d):
    """errorest of an oscillatory integral of one short list"""
    with pg.Workspace(d, 0) as ws:
        r = ws.integrate_genz("oscillatory", *_params("oscillatory", d), epsrel=1e-2, epsabs=1e-20)
    return [r.errorest.hex()]


def evaluated(pg, fam, d, precision, slices):
    """The exact sums of the estimates and errors of 321 regions"""
    import torch
    n = 321
    rng = np.random.default_rng(d)
    H = 0.5 ** rng.integers(1, 6, size=(d, n))
    L = np.floor(rng.random((d, n)) / H) * H
    dev = [torch.from_numpy(np.ascontiguousarray(x.ravel())).to("cuda:0") for x in (L, H)]
    est = torch.empty(n, dtype=torch.float64, device="cuda:0")
    err, dim = torch.empty_like(est), torch.empty(n, dtype=torch.uint8, device="cuda:0")
    with pg.Workspace(d, 0) as ws:
        ws.set_slices(slices)
        ws.eval_genz(fam, *_params(fam, d), n, *dev, est, err, dim, precision=precision)
    return [math.fsum(x.cpu().tolist()).hex() for x in (est, err)]


EVALS = [("oscillatory", 64, 1), ("oscillatory", 64, 4)] + [
    (f, 32, s) for f in ("oscillatory", "product_peak", "corner_peak", "gaussian", "c0", "discontinuous")
    for s in (1, 4)]

SEGMENTS = {
    2: ["0x1.021d46fa4d5b8p-40", "0x1.021d46fa4d5b8p-40"],
    3: ["0x1.a1770e5958866p-37", "0x1.a1770e5958866p-37"],
    4: ["0x1.0d5866bd20f20p-35", "0x1.0d5866bd20f20p-35"],
    5: ["0x1.7e58e05fb80fap-31", "0x1.7e58e05fb80fap-31"],
    6: ["0x1.5599b5dc1981fp-27", "0x1.5599b5dc1981fp-27"],
    8: ["0x1.feadc98cffedep-26", "0x1.feadc98cffedep-26"],
    10: ["0x1.23458138c747dp-24", "0x1.23458138c747dp-24"],
}
SHORT = {
    2: ["0x1.021ce7e53caa0p-40"],
    3: ["0x1.a1770f762eb0cp-37"],
    4: ["0x1.0d586714c5d28p-35"],
    5: ["0x1.7e58e08563950p-31"],
    6: ["0x1.5599b5dcc1411p-27"],
    8: ["0x1.feadc98cffedep-26"],
    10: ["0x1.23458138ca926p-24"],
}
EVAL = {
    ("c0", 32, 1): {
        2: ["0x1.f05ee4ff9070dp-2", "0x1.cc4ab5d4494b7p-3"],
        3: ["0x1.2643d6f16f9e3p-7", "0x1.7b7af31e27199p-8"],
        5: ["0x1.7aa49197c0192p-16", "0x1.7324ec2bbdb7cp-18"],
        8: ["0x1.680ef71eb92ebp-30", "0x1.ba9f463cfdf2dp-33"],
    },
    ("c0", 32, 4): {
        2: ["0x1.f05ee60434f27p-2", "0x1.cc4afd21baedbp-3"],
        3: ["0x1.2643d5fd12e6fp-7", "0x1.7b7af1db458e9p-8"],
        5: ["0x1.7aa490b881ed2p-16", "0x1.7324f3b8a36f6p-18"],
        8: ["0x1.680efa1cc5e2fp-30", "0x1.ba9f46fa0c37ap-33"],
    },
    ("corner_peak", 32, 1): {
        2: ["0x1.74c82f31cfb7cp-5", "0x1.6b5171686e1a1p-7"],
        3: ["0x1.a5e076e40a45dp-11", "0x1.feae76e0b2e0ap-12"],
        5: ["0x1.dbb48f643e079p-30", "0x1.40955286d04a4p-32"],
        8: ["0x1.3dd112ae52de8p-57", "0x1.b8ad76ccdc02ap-72"],
    },
    ("corner_peak", 32, 4): {
        2: ["0x1.74c82f6b52df0p-5", "0x1.6b51526e80e2bp-7"],
        3: ["0x1.a5e076e04b7bbp-11", "0x1.feae749b7ac2ap-12"],
        5: ["0x1.dbb48cbc3bffcp-30", "0x1.40953e69176d8p-32"],
        8: ["0x1.3dd116726e87dp-57", "0x1.b8d4bf6a107c2p-72"],
    },
    ("discontinuous", 32, 1): {
        2: ["0x1.acbf7ae5647d9p+11", "0x1.4c6e09fc6cec4p+12"],
        3: ["0x1.b5f1e111e3b15p+14", "0x1.078276166bce4p+15"],
        5: ["0x1.e2d6722d2a3a2p+9", "0x1.274166a16c9f3p+9"],
        8: ["0x1.3078f5bc52655p+15", "0x1.f81aa90b31521p+11"],
    },
    ("discontinuous", 32, 4): {
        2: ["0x1.acbf7ed7f4f96p+11", "0x1.4c6e0fac646c7p+12"],
        3: ["0x1.b5f1dcae3bfaep+14", "0x1.078270daa60e0p+15"],
        5: ["0x1.e2d67202a48ecp+9", "0x1.274172c01b3aep+9"],
        8: ["0x1.3078ca7f66977p+15", "0x1.f81a0bacbfdacp+11"],
    },
    ("gaussian", 32, 1): {
        2: ["0x1.0f19571a1099dp-2", "0x1.2f3922bb06b4ep-2"],
        3: ["0x1.ba7d5d4cc3522p-7", "0x1.162d8e5ccddd6p-7"],
        5: ["0x1.4898eeda71bedp-15", "0x1.029548e481687p-15"],
        8: ["0x1.cb4bd57db1c53p-42", "0x1.07bd9872f972ep-42"],
    },
    ("gaussian", 32, 4): {
        2: ["0x1.0f1956d7c0a62p-2", "0x1.2f392706aac79p-2"],
        3: ["0x1.ba7d5da32d3b2p-7", "0x1.162d8af8567d8p-7"],
        5: ["0x1.4898f70d2644cp-15", "0x1.02954fa7874c4p-15"],
        8: ["0x1.cb4c061bd24abp-42", "0x1.07bdb6586e6b0p-42"],
    },
    ("oscillatory", 32, 1): {
        2: ["-0x1.013d3a206cc29p+3", "0x1.0665ba4af6a92p-12"],
        3: ["0x1.5637f481101c8p+0", "0x1.1a58e98bc481ap-17"],
        5: ["0x1.161ff991b26abp-4", "0x1.d3b74d9926256p-23"],
        8: ["-0x1.058fcb34554c2p-13", "0x1.cef8b8189903cp-33"],
    },
    ("oscillatory", 32, 4): {
        2: ["-0x1.013d3a34bbd83p+3", "0x1.fbd4bee780de4p-12"],
        3: ["0x1.5637f4d66850dp+0", "0x1.a4a57f14dee80p-13"],
        5: ["0x1.161ff9f2a5001p-4", "0x1.758a251fb30f7p-18"],
        8: ["-0x1.058fcbce62ebep-13", "0x1.eabc2b22f9cfdp-24"],
    },
    ("oscillatory", 64, 1): {
        2: ["-0x1.013d3a03c9820p+3", "0x1.a923d31fba5e6p-32"],
        3: ["0x1.5637f3379e6b3p+0", "0x1.f82f73ab39962p-30"],
        5: ["0x1.161ffa32dada5p-4", "0x1.2e7c61ae5014ap-33"],
        8: ["-0x1.058fc659af70dp-13", "0x1.9e7239dbe2616p-43"],
    },
    ("oscillatory", 64, 4): {
        2: ["-0x1.013d3a03c9820p+3", "0x1.a923d7088db22p-32"],
        3: ["0x1.5637f3379e6b3p+0", "0x1.f82f736d1430fp-30"],
        5: ["0x1.161ffa32dada5p-4", "0x1.2e7c618754e5ap-33"],
        8: ["-0x1.058fc659af70ep-13", "0x1.9e723a296bcffp-43"],
    },
    ("product_peak", 32, 1): {
        2: ["0x1.74a71fe3ddf86p+12", "0x1.368936438c284p+10"],
        3: ["0x1.7b64a087a8789p+15", "0x1.d6241c9f82f92p+13"],
        5: ["0x1.2e858dea5c323p+18", "0x1.fadc1f96b13acp+15"],
        8: ["0x1.d155fe87efc3ap+27", "0x1.fdfe17db0d58fp+24"],
    },
    ("product_peak", 32, 4): {
        2: ["0x1.74a71f12dfb3dp+12", "0x1.3688ba6626ed6p+10"],
        3: ["0x1.7b64a05e518c1p+15", "0x1.d6241ddb4a77ap+13"],
        5: ["0x1.2e858dd77c23cp+18", "0x1.fadc1d7f17ea7p+15"],
        8: ["0x1.d1560079ffc80p+27", "0x1.fdfe20e6a0550p+24"],
    },
}


@pytest.mark.parametrize("d", DIMS)
def test_oscillatory_segments(pg, gpu, d):
    assert segments(pg, d) == SEGMENTS[d]


@pytest.mark.parametrize("d", DIMS)
def test_oscillatory_short_list(pg, gpu, d):
    assert short_list(pg, d) == SHORT[d]


@pytest.mark.parametrize("fam,precision,slices", EVALS)
def test_evaluated(pg, gpu, fam, precision, slices):
    got = {d: evaluated(pg, fam, d, precision, slices) for d in (2, 3, 5, 8)}
    assert got == EVAL[fam, precision, slices]
