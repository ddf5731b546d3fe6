"""QL of batches that LDS holds only a part of at a time (rows in device memory):
the oracle's bits around the sizes where the rows change place and past a round of
wavefronts, the tridiagonal that does not converge named, outputs that are the
inputs, and a cost a rule that does not grow with the batch.

Bar: the same bits; the 32768 rules of n = 256 within five times the call of 2048
(chains run side by side: 2.0 measured, 9.3 with the rows in LDS)."""
import time

import numpy as np
import pytest
import torch

from conftest import MG1

import sqminiapp_amd as sq

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def ctx():
    c = sq.Context(MG1, "Mg1", phantom_atom=True, device=0)
    yield c
    c.close()


def _tridiags(n, count):
    rng = np.random.default_rng(n + count)
    return rng.uniform(-1, 25, (count, n)), rng.uniform(0.5, 9, (count, n))


@pytest.mark.parametrize("n,count", [(106, 16384), (106, 16385), (107, 4096), (107, 4097), (171, 2049), (256, 2049),
                                     (1, 16390), (7, 131072 + 70)])
def test_rules_bit_identical_to_the_oracle(ctx, oracle_mod, n, count):
    d, s = _tridiags(n, count)
    s[::3, n // 2] = 0.0   # a split in every third
    lam, w, lmin, lmax = ctx.tridiag_nodes_weights(d, s)
    for r in sorted({0, 1, 63, 64, count // 2, count - 70, count - 2, count - 1}):
        lo, wo, mn, mx = oracle_mod.tridiag_nodes_weights(d[r], s[r], n)
        assert np.array_equal(lam[r], lo) and np.array_equal(w[r], wo) and lmin[r] == mn and lmax[r] == mx, r
    rows = np.arange(0, count, max(1, count // 50))
    one = ctx.tridiag_nodes_weights(d[rows], s[rows])
    assert np.array_equal(lam[rows], one[0]) and np.array_equal(w[rows], one[1])


def test_failed_tridiagonal_and_outputs_in_place(ctx):
    n, count = 10, 30000
    d, s = _tridiags(n, count)
    ref = ctx.tridiag_nodes_weights(d, s)
    dd, ds = (torch.from_numpy(x).to("cuda:0") for x in (d, s))
    ends = [torch.empty(count, dtype=torch.float64, device="cuda:0") for _ in range(2)]
    torch.cuda.synchronize()
    ctx.tridiag_nodes_weights_noalloc(dd.data_ptr(), ds.data_ptr(), n, count, dd.data_ptr(), ds.data_ptr(),
                                      *(t.data_ptr() for t in ends))
    for got, want in zip((dd, ds, *ends), ref):
        assert np.array_equal(got.cpu().numpy(), want)
    d[29000, 3] = np.nan
    with pytest.raises(sq.SQError, match="29000"):
        ctx.tridiag_nodes_weights(d, s)


def test_a_large_batch_costs_no_more_a_rule(ctx):
    ms = []
    for count in (2048, 32768):
        d, s = _tridiags(256, count)
        best = np.inf
        for _ in range(3):
            t = time.perf_counter()
            ctx.tridiag_nodes_weights(d, s)
            best = min(best, time.perf_counter() - t)
        ms.append(1e3 * best)
    print(f"n = 256: 2048 rules {ms[0]:.1f} ms, 32768 rules {ms[1]:.1f} ms", flush=True)
    assert ms[1] < 5 * ms[0]
