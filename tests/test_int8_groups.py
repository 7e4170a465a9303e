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
