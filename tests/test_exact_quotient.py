"""The quantizer's division-free quotient (RN(1/s), product, exact residual,
correction) against IEEE division, in numpy: float64 holds every intermediate
of the two fused operations exactly before their rounding to float32."""

from __future__ import annotations

import numpy as np
import pytest


def _quotient(x, s):
    r = np.float32(1.0) / s
    q0 = x * r
    wide = np.float64
    residual = (x.astype(wide) - q0.astype(wide) * s.astype(wide)).astype(np.float32)
    return (q0.astype(wide) + residual.astype(wide) * r.astype(wide)).astype(np.float32)


def _check(x, s):
    got, want = _quotient(x, s), x / s
    assert np.array_equal(got, want), int((got != want).sum())


@pytest.mark.parametrize("spread", [1e-6, 1.0, 6e4])
def test_random_differences_of_halves(spread):
    rng = np.random.default_rng(7)
    half = lambda: (rng.standard_normal(400_000) * spread).clip(-65504, 65504).astype(np.float16)  # noqa: E731
    x = half().astype(np.float32) - half().astype(np.float32)
    page = np.abs(x).reshape(-1, 16).max(axis=1) / np.float32(127.0)
    s = np.maximum(page, np.float32(2.0 ** -20)).astype(np.float16).astype(np.float32)
    _check(x.reshape(-1, 16), s[:, None])


def test_every_scale_mantissa_near_code_boundaries():
    # every 11-bit scale mantissa, x next to (code + 1/2) * s
    s = (np.arange(1024, 2048, dtype=np.float32) * np.float32(2.0 ** -14))[:, None]
    boundary = ((np.arange(0, 127, dtype=np.float64) + 0.5)[None, :] * s).astype(np.float32)
    for ulps in (-2, -1, 0, 1, 2):
        x = boundary
        for _ in range(abs(ulps)):
            x = np.nextafter(x, np.float32(np.inf if ulps > 0 else -np.inf), dtype=np.float32)
        _check(x, np.broadcast_to(s, x.shape))
