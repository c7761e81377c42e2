"""The batched event kernel at the edges of its units: 1 to 8 groups of 8 starts
(one to two half groups share a unit's events between the waves, three to four take
them whole), wave counts with a padded last block, and bins of one ragged tile, a
whole tile, one event more and several chunks.  Against the oracle with the
tolerances of test_gpu_batch.py, and bitwise: a fit's value and gradient do not
depend on how many other starts its unit holds."""
import numpy as np
import pytest

from tests import test_gpu_batch as TB

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("waves,starts", [(1, 1), (3, 8), (7, 9), (8, 16), (9, 17), (16, 24), (23, 25), (40, 33), (88, 64),
                                          # every swizzle of the rows (padded waves / 8 odd, even, a multiple of
                                          # 4) in both kinds of unit, up to the most waves
                                          (25, 12), (32, 57), (48, 45), (56, 20), (64, 16), (72, 10), (80, 56),
                                          (89, 13), (96, 64)])
def test_edges(gpu, waves, starts):
    bins = TB.make_bins(waves, [31, 32, 33, 1025], seed=320 + waves)
    par = TB.fp32_params(np.random.default_rng(waves), len(bins), starts, 2 * waves, 2.0)
    v, g = TB.check_against_oracle(TB.make_batch(waves, starts, bins), bins, par, starts=sorted({0, starts // 2, starts - 1}))
    for first, n in ((0, 1), (starts // 2, starts - starts // 2)):
        v2, g2 = TB.make_batch(waves, n, bins).eval(np.ascontiguousarray(par[:, first:first + n]))
        assert np.array_equal(v2, v[:, first:first + n])
        assert np.array_equal(g2, g[:, first:first + n])
