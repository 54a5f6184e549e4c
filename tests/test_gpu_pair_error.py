"""Rounding error of the full-FP64 tiled path's pair terms, against extended precision and the plain FP64 path.

Two atoms on the x axis at distances with few bits, charges and LJ parameters large enough that the fixed-point sums hold
every bit of a term: what is measured is the pair arithmetic alone.  Errors are in units of 2^-53 of the term's undamped,
unswitched magnitude, as root mean squares over the distances of a range.  The plain path evaluates the reference's
expressions (pMolecule-1.9.0/extensions/cinclude/PairwiseInteraction.h:72-119: divide and square root).

The bound: no range's error above 1.25 times the plain path's, plus 0.25 units.  On the CPU, with the same forms and a
seed off by up to 2^-23, the ratios are at most 1.07 (below 1 in most ranges); the root mean squares of 200 samples
scatter by some 5% each, and the product of the force with the distance adds 0.3 units to either side.  The same forms
with 1/r left 2 units off and the switched Lennard-Jones squares expanded give ratios of 1.6 to 4.
"""

import math

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

LD = np.longdouble
# Angstrom up to the inner cutoff (None), then fractions of the switched range.
RANGES = [(0.6, 2.0), (2.0, 2.8), (2.8, 3.5), (3.5, 5.0), (5.0, None)]
SWITCHED = [(0.0, 0.5), (0.5, 0.8), (0.8, 0.997)]
SAMPLES = 200


def _exact(r, qq, A, B, inner, outer):
    """(Coulomb, LJ, Coulomb and LJ dE/dr) of one pair beyond the damping radius, and their scales, in extended precision."""
    r, qq, A, B, on, off = (LD(v) for v in (r, qq, A, B, inner, outer))
    r2, on2, off2 = r * r, on * on, off * off
    gamma = (off2 - on2) ** 3
    a, b, c, d = off2 * off2 * (off2 - 3 * on2) / gamma, 6 * off2 * on2 / gamma, -(off2 + on2) / gamma, LD(2) / 5 / gamma
    q1 = 8 * (off2 * on2 * (off - on) - (off * off2 * off2 - on * on2 * on2) / 5) / gamma
    q2 = -a / off + b * off + c * off * off2 + d * off * off2 * off2
    s = 1 / r
    s3 = s * s * s
    s6 = s3 * s3
    if r2 > on2:
        el = qq * (s * (a - r2 * (b + r2 * (c + d * r2))) + q2)
        fe = -qq * s * (a + r2 * (b + r2 * (3 * c + 5 * d * r2))) * s
        l1, l2 = s6 - 1 / off2 ** 3, s3 - 1 / (off * off2)
        kA, kB = A * off2 ** 3 / (off2 ** 3 - on2 ** 3), B * off * off2 / (off * off2 - on * on2)
        lj = kA * l1 * l1 - kB * l2 * l2
        fl = -12 * kA * l1 * s6 * s + 6 * kB * l2 * s3 * s
    else:
        el, fe = qq * (s + q1), -qq * s * s
        lj = A * (s6 * s6 - 1 / (on * off) ** 6) - B * (s6 - 1 / (on * off) ** 3)
        fl = (-12 * A * s6 * s6 + 6 * B * s6) * s
    return (el, lj, fe, fl), (abs(qq) * s, A * s6 * s6 + B * s6, abs(qq) * s * s, (12 * A * s6 * s6 + 6 * B * s6) * s)


def _errors(precision, inner, outer, lo, hi, seed):
    from pdynamo_amd import NBModelABFS, _native
    rng = np.random.default_rng(seed)
    factor = (1.0e+7 * 6.0221415e+23 * 1.60217653e-19 * 1.60217653e-19) / (4.0 * math.pi * 8.854187817e-12)
    # escale = factor / dielectric = 2^20, so the product of the charges is exact on either path.
    model = NBModelABFS(precision=precision, dielectric=factor / 2.0 ** 20, innerCutoff=inner, outerCutoff=outer,
                        listCutoff=outer + 1.5)
    q = np.array([4096.0 * 1.25, -4096.0 * 0.8125])
    eps, sigma = (2.0 ** 24 if lo < 2.0 else 2.0 ** 50), 3.15
    A, B = 4.0 * eps * sigma ** 12, 4.0 * eps * sigma ** 6
    coulomb = _native.NativeState(model.NativeOptions(), q, np.zeros(2, np.int32), 1, np.zeros(1), np.zeros(1))
    lj = _native.NativeState(model.NativeOptions(), np.zeros(2), np.zeros(2, np.int32), 1, np.array([A]), np.array([B]))
    qq = q[0] * q[1] * 2.0 ** 20
    out = []
    for _ in range(SAMPLES):
        r = round(rng.uniform(lo, hi) * 65536.0) / 65536.0
        x = np.array([[0.0, 0.0, 0.0], [r, 0.0, 0.0]])
        got = []
        for st, term in ((coulomb, 0), (lj, 1)):
            g = np.zeros((2, 3))
            e, _, _ = st.energy_host(x, g)
            got.append((e[term], g[1, 0]))
            assert g[0, 0] == -g[1, 0]
        ref, scale = _exact(r, qq, A, B, inner, outer)
        val = (got[0][0], got[1][0], got[0][1], got[1][1])
        out.append([float((LD(v) - w) / s) * 2.0 ** 53 for v, w, s in zip(val, ref, scale)])
    coulomb.close()
    lj.close()
    return np.sqrt((np.array(out) ** 2).mean(0))


@pytest.mark.parametrize("k", range(len(RANGES) + len(SWITCHED)))
@pytest.mark.parametrize("inner,outer", [(8.0, 12.0), (7.0, 11.0)])
def test_full_fp64_pair_terms_as_exact_as_the_reference_expressions(inner, outer, k):
    if k < len(RANGES):
        lo, hi = RANGES[k][0], RANGES[k][1] or inner
    else:
        lo, hi = (inner + f * (outer - inner) for f in SWITCHED[k - len(RANGES)])
    tiled = _errors("tiled_fp64", inner, outer, lo, hi, 100 + k)
    plain = _errors("fp64", inner, outer, lo, hi, 100 + k)
    print("%.2f-%.2f A: tiled %s, plain %s" % (lo, hi, np.round(tiled, 2), np.round(plain, 2)), flush=True)
    assert (tiled <= 1.25 * plain + 0.25).all(), (tiled, plain)
