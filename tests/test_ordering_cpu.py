"""CPU checks that the tiled kernel's results cannot depend on the order of its work items.

The fixed-point sums (``fx_split``/``fx_value`` in csrc/nbabfs_internal.h) decide this, restated here in numpy: every
force and energy contribution becomes two int64 words, hi = rint(v / 2^16) and lo = rint((v - hi 2^16) 2^32), added with
integer atomics.  Integer addition is associative, so any order of the items gives the same words, and the words convert
to the same double.  An item's energy is added as twice its value, with twice the range.

The plain FP64 path adds in FP64: its rows do not read work items (one thread per atom over sorted CSR rows), and its
image items keep one order (tests/test_gpu_images.py).  How items are cut and laid out: tests/test_item_rules_cpu.py.
"""

import numpy as np

HI_UNIT = 2.0 ** 16
LO_SCALE = 2.0 ** 32


def fx_split(v, limit=2.0 ** 66):
    v = np.clip(v, -limit, limit)
    hi = np.rint(v / HI_UNIT)
    r = v - hi * HI_UNIT                     # exact (Sterbenz: |r| <= 2^15)
    lo = np.rint(r * LO_SCALE)
    return hi.astype(np.int64), lo.astype(np.int64)


def fx_value(hi, lo):
    return float(hi) * HI_UNIT + float(lo) / LO_SCALE


def test_fixed_point_sums_do_not_depend_on_item_order():
    rng = np.random.default_rng(3)
    # contributions of many items to one gradient component: ordinary forces and a few overlaps
    v = rng.normal(0.0, 50.0, 20000) * np.where(rng.random(20000) < 0.01, 1e9, 1.0)
    hi, lo = fx_split(v)
    ref = (int(hi.sum()), int(lo.sum()))
    for seed in range(5):
        p = np.random.default_rng(seed).permutation(v.size)
        h2, l2 = fx_split(v[p])
        assert (int(h2.sum()), int(l2.sum())) == ref
    # each contribution is represented to half a unit of 2^-32
    back = hi.astype(np.float64) * HI_UNIT + lo.astype(np.float64) / LO_SCALE
    small = np.abs(v) < 2.0 ** 20
    assert np.max(np.abs(back[small] - v[small])) <= 2.0 ** -32


def test_item_energies_keep_their_range_and_rounding():
    """Twice an item's energy: up to 2^66 kJ/mol is inside the range, the sum of 4,096 such items stays inside int64, and
    an ordinary item's energy is held to 2^-34 kJ/mol, so that four times the items round to the error of one split."""
    rng = np.random.default_rng(8)
    e = np.concatenate([rng.uniform(-1.0, 1.0, 4094) * 2.0 ** 66, [2.0 ** 66, -2.0 ** 66]])
    hi, lo = fx_split(2.0 * e, 2.0 ** 67)
    assert np.abs(hi).max() == 2 ** 51 and abs(sum(int(h) for h in hi)) < 2 ** 63
    for h, l, v in zip(hi, lo, e):
        assert 0.5 * fx_value(int(h), int(l)) == v
    e = rng.normal(0.0, 300.0, 20000)
    hi, lo = fx_split(2.0 * e, 2.0 ** 67)
    back = 0.5 * (hi.astype(np.float64) * HI_UNIT + lo.astype(np.float64) / LO_SCALE)
    assert np.max(np.abs(back - e)) <= 2.0 ** -34
    words = {(int(hi[p].sum()), int(lo[p].sum())) for p in (np.random.default_rng(k).permutation(e.size) for k in range(5))}
    assert len(words) == 1
