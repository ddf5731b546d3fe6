"""The resident Lanczos kernel (FP64, one node a workgroup, its vectors on chip)
against the column-marching kernels it stands before, over the shapes that
select its builds: cubes below and above 512 columns, plane counts at and
between the unrolled sizes, sides that differ, vectors that fit LDS whole and
not, both operators, node ranges that start anywhere.

SQ_NO_RESIDENT runs the column-marching kernels.  Bar: the two sum the same
terms in another order, so tridiagonals agree to 1e-10 of the spectrum's
width after a few steps (the existing kernels' bar against the oracle).
"""
import numpy as np
import pytest

import sqminiapp_amd as sq
from sqminiapp_amd import decks

pytestmark = pytest.mark.gpu

# (repetitions, spacing, truncation radius): nloc 17^3, 21^3 (512 threads), 25^3, 29^3 and 31 planes (1024)
SHAPES = [((1, 1, 1), 0.75, 6.0), ((1, 1, 1), 0.6, 6.0), ((2, 1, 1), 0.55, 6.5), ((1, 1, 1), 0.5, 7.0),
          ((1, 1, 2), 0.5, 7.4)]


def _deck(tmp_path, reps, h, rcut, nqp):
    cfg = decks.Supercell("cell", reps, sigma=0.15, seed=7, h_target=h, rcut=rcut, nqp=nqp)
    return decks.write_deck(cfg, str(tmp_path / f"{reps}_{h}_{rcut}")), cfg.name


@pytest.mark.parametrize("reps,h,rcut", SHAPES)
def test_resident_matches_the_column_marching_kernels(monkeypatch, tmp_path, reps, h, rcut):
    d, name = _deck(tmp_path, reps, h, rcut, 8)
    res = {}
    for off in (False, True):
        monkeypatch.setenv("SQ_NO_RESIDENT", "1") if off else monkeypatch.delenv("SQ_NO_RESIDENT", raising=False)
        with sq.Context(d, name) as c:
            planes = c.resident_planes()
            assert (planes == 0) == off
            n = c.n_nodes
            veff = np.random.default_rng(11).normal(0.3, 0.2, tuple(c.info.npts)[::-1])
            c.set_veff(veff)
            for mode in (sq.SQ_NL_KB, sq.SQ_NL_REF_COLLAPSED):
                for begin, count in ((0, 1), (n - 3, 3), (n // 3 + 5, 65)):
                    c.run(mode, sq.SQ_FP64, begin=begin, count=count)
                    res[off, mode, begin] = c.lanczos()
            nloc = tuple(c.info.nloc)
    for key in [k for k in res if not k[0]]:
        (a, b), (a0, b0) = res[key], res[(True,) + key[1:]]
        width = np.abs(a0).max() + 2 * np.abs(b0).max()
        err = max(np.abs(a - a0).max(), np.abs(b - b0).max()) / width
        print(f"nloc {nloc} mode {key[1]} from {key[2]}: {err:.2e}", flush=True)
        assert err < 1e-10


def test_resident_forces_match_the_column_marching_kernel(monkeypatch, tmp_path):
    """The force pass records the same alphas: nonlocal forces of one SCF pass in both kernels."""
    d, name = _deck(tmp_path, (1, 1, 1), 0.6, 6.0, 10)
    f = {}
    for off in (False, True):
        monkeypatch.setenv("SQ_NO_RESIDENT", "1") if off else monkeypatch.delenv("SQ_NO_RESIDENT", raising=False)
        with sq.Context(d, name, cell=True) as c:
            c.scf(sq.SQ_NL_KB, sq.SQ_FP64, max_iter=1)
            f[off] = c.forces()[2]
    assert np.abs(f[True]).max() > 1e-4
    assert np.abs(f[False] - f[True]).max() < 1e-9
