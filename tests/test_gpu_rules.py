"""The QL kernel's rules bit for bit against the oracle where its launch or its
arithmetic takes another form: batches below and above one wavefront a CU,
row counts that lower the tridiagonals of a wavefront, and entries of a size
at which a rotation falls back to the operators.

Bar: the same bits; a rule may not depend on the batch it was part of either.
"""
import numpy as np
import pytest

from conftest import MG1

import sqminiapp_amd as sq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = sq.Context(MG1, "Mg1", phantom_atom=True, device=0)
    yield c
    c.close()


@pytest.mark.parametrize("n,count,scale", [(1, 3, 1.0), (2, 257, 1.0), (80, 256, 1.0), (80, 4097, 1.0), (80, 8193, 1.0),
                                           (86, 8192, 1.0), (120, 5000, 1.0), (256, 1100, 1.0), (40, 70, 2.0 ** -340),
                                           (40, 70, 2.0 ** 340)])
def test_rules_bit_identical_to_the_oracle(ctx, oracle_mod, n, count, scale):
    rng = np.random.default_rng(n + count)
    d = rng.uniform(-1, 25, (count, n)) * scale
    s = rng.uniform(0.5, 9, (count, n)) * scale
    s[::3, n // 2] = 0.0   # a split in every third
    lam, w, lmin, lmax = ctx.tridiag_nodes_weights(d, s)
    for r in sorted({0, 1, count // 2, count - 2, count - 1}):
        lo, wo, mn, mx = oracle_mod.tridiag_nodes_weights(d[r], s[r], n)
        assert np.array_equal(lam[r], lo) and np.array_equal(w[r], wo) and lmin[r] == mn and lmax[r] == mx, r
    rows = np.arange(0, count, max(1, count // 50))
    one = ctx.tridiag_nodes_weights(d[rows], s[rows])
    assert np.array_equal(lam[rows], one[0]) and np.array_equal(w[rows], one[1])
