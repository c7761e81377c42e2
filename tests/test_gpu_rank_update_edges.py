"""The rank-k updates of the integral and of the Hessian at the edges of their
geometry: rows of 1 column block of 8 waves, of one window (12 and 11 blocks) and
of two and three windows (up to 8 blocks) with a padded last block, single events,
chunks of up to 64 events with a ragged last one, and several chunks per workgroup.

Reference: numpy.  Both sides sum M terms in FP64, in different orders: the
difference from a sum is below M 2^-53 relative to the sum of magnitudes, with M up
to 33k 4e-12 in the worst case and its square root (2e-14) as it happens; 1e-12
relative to the largest element, as the other integral tests."""
import numpy as np
import pytest

from tests import helpers as H

pytestmark = pytest.mark.gpu


def amplitudes(rng, M, W):
    return (rng.normal(size=(M, W)) + 1j * rng.normal(size=(M, W))) * np.linspace(0.4, 1.6, W)[None, :]


@pytest.mark.parametrize("waves,events", [(1, 1), (7, 63), (8, 64), (9, 65), (16, 7), (24, 129), (87, 55), (88, 57),
                                          (89, 111), (96, 8), (97, 56), (104, 64), (128, 65), (137, 64 * 256 * 2 + 9)])
def test_integral(gpu, waves, events):
    rng = np.random.default_rng(waves)
    a = amplitudes(rng, events, waves)
    w = rng.uniform(0.5, 2.0, size=events)
    assert H.rel_err(gpu.integral(a), a.T @ a.conj()) <= 1e-12
    ref = (a / w[:, None]).T @ a.conj() * (events / np.sum(1 / w))
    assert H.rel_err(gpu.integral(a, w), ref) <= 1e-12
