"""The density network's kernels at the edges of their tiles: descriptors on
cells that are no whole number of bricks, and on a dense cell whose image list is
taken in more than one piece; gradient sums for row counts around the tile and the
chunk, repeated with a workspace of another size in between; the guess on one
device against descriptors and forward one after the other.

Bars: descriptors as stored in FP32 (1e-6 of the largest); gradient sums as for
any count (FP32 activations, double sums: 1e-4 of the largest, the loss to 1e-5).
"""
import numpy as np
import pytest

from oracle import mlp as M

import sqminiapp_amd as sq
from sqminiapp_amd import decks

pytestmark = pytest.mark.gpu
K, H = 32, 64


@pytest.mark.parametrize("reps,a,c,h", [((1, 1, 1), 6.06, 9.83, 1.6), ((2, 1, 1), 6.06, 9.83, 0.77),
                                        ((3, 2, 2), 3.5, 5.7, 1.4)])
def test_descriptors_at_brick_and_list_edges(tmp_path, reps, a, c, h):
    cfg = decks.Supercell("cell", reps, a=a, c=c, sigma=0.1, seed=3, h_target=h, rcut=4.0, nqp=4)
    with sq.Context(decks.write_deck(cfg, str(tmp_path)), cfg.name, cell=True) as ctx:
        f = ctx.descriptors()
        I = ctx.info
        G = (I.npts[0] - 1, I.npts[1] - 1, I.npts[2] - 1)
        ref = M.features(cfg.positions(), list(I.delta), list(I.range), G)
        assert f.shape == ref.shape and np.max(np.abs(f - ref)) < 1e-6 * max(1.0, np.max(np.abs(ref)))
        with sq.Mlp(seed=2) as m:
            guess = m.guess(ctx)
            p, norm = m.params()
            y = m.forward(f.reshape(-1, K))
            rat = ctx.cell_field("rho_atomic")
            want = np.maximum(0.0, rat + float(norm[-1]) * y.reshape(rat.shape).astype(np.float64))
            want *= I.noetot / (want.sum() * I.dV)
            assert np.max(np.abs(guess - want)) < 1e-12 * np.max(np.abs(want))


def test_gradient_at_tile_and_chunk_edges():
    rng = np.random.default_rng(8)
    first = {}
    with sq.Mlp(seed=5) as m:
        p = m.params()[0].astype(np.float64)
        for n in (1, 31, 32, 33, 64, 8191, 8192, 8225, 33, 9000, 1):
            x = np.random.default_rng(n).normal(0, 1, (n, K)).astype(np.float32)
            t = np.random.default_rng(n + 1).normal(0, 1, n).astype(np.float32)
            L, g = m.loss_grad(x, t)
            L_ref, g_ref = M.loss_grad(p, x.astype(np.float64), t.astype(np.float64), K, H)
            assert L == pytest.approx(L_ref, rel=1e-5), n
            assert np.max(np.abs(g - g_ref)) < 1e-4 * np.max(np.abs(g_ref)), n
            if n in first:   # the same bits from a workspace used for other counts
                assert L == first[n][0] and np.array_equal(g, first[n][1])
            first[n] = (L, g.copy())
