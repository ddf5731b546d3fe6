"""The resident kernel against the oracle on cubes whose sides differ, in each of its
builds and with plane counts below a build's: an x for a y or a z in a column,
a table or the halo shows there and not on a cube of equal sides.  And where it
hands over: a side past 31 points, or a cube that meets more than 128 images.

Bar: tridiagonals to 1e-10 of the spectrum's width after eight steps, random
potential, both operators (the kernels' bar against the oracle).
"""
import numpy as np
import pytest

import sqminiapp_amd as sq
from sqminiapp_amd import decks

pytestmark = pytest.mark.gpu

# (a, c, spacing, truncation radius), the cube, whether the kernel holds it
SHAPES = [((5.2, 9.83, 0.75, 7.0), (19, 21, 21), True),    # 512 threads, 21 planes
          ((6.06, 8.9, 0.75, 7.0), (21, 19, 19), True),
          ((5.2, 9.83, 0.66, 7.4), (21, 23, 23), True),    # 512 threads, 25 planes
          ((6.06, 9.83, 0.66, 7.0), (23, 23, 21), True),   # 1024 threads, 25 planes
          ((5.2, 9.83, 0.57, 6.5), (25, 23, 25), True),
          ((5.2, 9.83, 0.57, 7.0), (27, 25, 27), True),    # 1024 threads, 29 planes
          ((6.6, 9.83, 0.55, 7.4), (29, 27, 27), True),
          ((5.2, 9.83, 0.48, 7.0), (29, 29, 31), True),    # 1024 threads, 31 planes
          ((4.8, 8.0, 0.6, 6.0), (21, 21, 21), True),      # 115 images a cube
          ((4.8, 7.8, 0.6, 6.0), (21, 21, 21), False),     # 130
          ((5.6, 9.1, 0.55, 7.4), (29, 27, 29), False),    # 135
          ((5.2, 9.83, 0.48, 7.4), (31, 31, 33), False),
          ((5.6, 9.1, 0.48, 7.4), (31, 33, 31), False)]


@pytest.mark.parametrize("cell,nloc,held", SHAPES)
def test_lanczos_matches_the_oracle(tmp_path, oracle_mod, cell, nloc, held):
    a, c, h, rcut = cell
    cfg = decks.Supercell("cell", (1, 1, 1), a=a, c=c, sigma=0.15, seed=7, h_target=h, rcut=rcut, nqp=8)
    deck = decks.write_deck(cfg, str(tmp_path)), cfg.name
    S = oracle_mod.System(*deck)
    S.set_phantom(False)
    S.build_nonlocal()
    with sq.Context(*deck) as ctx:
        I = ctx.info
        assert tuple(I.nloc) == nloc and (ctx.resident_planes() > 0) == held and (I.batch[0] == 0) == held
        veff = np.random.default_rng(11).normal(0.3, 0.2, tuple(I.npts)[::-1])
        ctx.set_veff(veff)
        n, lx, ly = ctx.n_nodes, I.rank_box[3], I.rank_box[4]
        for mode in (sq.SQ_NL_KB, sq.SQ_NL_REF_COLLAPSED):
            for node in (0, n // 3 + 5, n - 1):
                ctx.run(mode, sq.SQ_FP64, begin=node, count=1)
                ab = np.array(ctx.lanczos())[:, 0]
                ref = np.array(S.lanczos((node // (lx * ly), node // lx % ly, node % lx), mode=mode, veff=veff))
                width = np.abs(ref[0]).max() + 2 * np.abs(ref[1]).max()
                err = np.abs(ab - ref).max() / width
                print(f"nloc {nloc} mode {mode} node {node}: {err:.2e}", flush=True)
                assert err < 1e-10
