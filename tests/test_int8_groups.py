"""GPU: the digit groups of the INT8-split bundle (three digits to an integer, 0..2, 3..5, 6).

Every count of digits, so every fill of a group, bit for bit against the numpy restatement that
adds digit by digit (oracle/int8_split.py): on rough data, where the mixed results of the last
digits use all their bits, on extents around one tile (28), and with values at a tie of the
last digit of a group.
"""
from __future__ import annotations

import numpy as np
import pytest

import int8_split as I8
from conftest import gpu_available
from test_int8 import hip_bundle

pytestmark = [pytest.mark.gpu,
              pytest.mark.skipif(not gpu_available(), reason="needs a HIP device")]


def rough_state(shape, seed):
    rng = np.random.default_rng(seed)
    F = rng.uniform(-1.0, 1.0, size=(24,) + tuple(shape))
    F[1] *= 2.0 ** rng.integers(-40, 40, size=shape)       # digits of all weights
    # multiples of half a unit of digit 2 and of digit 5, the field's range a power of two
    F[2] = np.rint(F[2] * 2.0 ** 21) * 2.0 ** -21
    F[3] = np.rint(F[3] * 2.0 ** 42) * 2.0 ** -42
    for f in (2, 3):
        F[f].flat[0], F[f].flat[-1] = 1.0, -1.0
    return F


@pytest.mark.parametrize("k", [1, 2, 3, 4, 5, 6, 7])
@pytest.mark.parametrize("shape", [(29, 7, 28), (6, 30, 27)])
def test_digit_groups_bitwise(k, shape):
    print(f"[case] digit groups k={k} {shape}", flush=True)
    F = rough_state(shape, seed=k)
    h = (0.07, 0.05, 0.11)
    got, want = hip_bundle(F, h, k), I8.bundle(F, h, k)
    assert np.array_equal(got, want), np.argwhere(got != want)[:5]


@pytest.mark.parametrize("k", [1, 2, 4, 7])
def test_infinite_values(k):
    """An infinity has no digits. In a tile with -inf the offset is -inf, every other value's
    difference is +inf, whose digit is -1 in the first place and 0 after it (the device's
    conversion), and the others' is 0; with +inf, or both, all digits are 0. So on the planes
    through it the bundle is that of a field of -1/64 with 0 at the infinity (the exponent of an
    infinity is 0, its scale 2^6), or of 0; every other plane's is its own."""
    print(f"[case] infinities k={k}", flush=True)
    shape, h = (9, 8, 10), (0.07, 0.05, 0.11)
    F = np.random.default_rng(k).uniform(-1.0, 1.0, size=(24,) + shape)
    bad, G = F.copy(), np.zeros_like(F)
    at = (4, 3, 6)
    for f, values in ((0, [-np.inf]), (4, [np.inf]), (9, [np.inf, -np.inf]), (12, [-np.inf])):
        for i, v in enumerate(values):
            bad[(f,) + (at if i == 0 else (4, 3, 2))] = v
        if values == [-np.inf]:
            G[f] = -1.0 / 64.0
            G[(f,) + at] = 0.0
    got, own, inf = hip_bundle(bad, h, k), I8.bundle(F, h, k), I8.bundle(G, h, k)
    for d in range(138):
        f = d // 3 if d < 72 else [0, 1, 3, 4, 5, 6, 7, 8, 9, 10, 11][(d - 72) // 6]
        # the axis along which the planes of this derivative are stacked
        axis = (1, 0, 0)[d % 3] if d < 72 else (1, 2, 1, 0, 0, 0)[(d - 72) % 6]
        want = own[d].copy()
        planes = [slice(None)] * 3
        if f in (0, 4, 9, 12):
            for q in {at[axis], (4, 3, 2)[axis] if f == 9 else at[axis]}:
                planes[axis] = q
                want[tuple(planes)] = inf[d][tuple(planes)]
        if f == 9 and axis == 2:       # the two infinities lie in different (x, y) planes
            planes[axis] = 2
            lone = np.zeros((24,) + shape)
            lone[9] = -1.0 / 64.0
            lone[9, 4, 3, 2] = 0.0
            want[tuple(planes)] = I8.bundle(lone, h, k)[d][tuple(planes)]
        assert np.array_equal(got[d], want), (d, np.argwhere(got[d] != want)[:5])
