"""SQ_BATCH, SQ_ZMARCH_WG and SQ_BATCH_TRIP choose the FP64 kernel where the
resident kernel would run too, and sq_info reports the kernel that runs: the
selection rule on the CPU, and on the device the same bits as with the resident
kernel left out altogether."""
import numpy as np
import pytest

from conftest import KERNEL_ENV, MG1, write_variant

import sqminiapp_amd as sq

FP64_AV = [1, 1, 1, 1, 0, 1]   # the resident kernel takes the last place


def test_resident_candidate_of_the_selection_rule():
    ms = [5.0, 4.0, 3.0, 6.0, 0.0, 2.0]
    sel = lambda ms, av=FP64_AV, **kw: sq.tune_select(sq.SQ_FP64, av, ms, **kw)  # noqa: E731
    assert sel(ms) == 5 and sel([5.0, 4.0, 3.0, 6.0, 0.0, 3.5]) == 2
    assert sel([5.0, 4.0, 3.0, 6.0, 0.0, 9.0], batch=0) == 5 and sel(ms, batch=0, trip=0) == 5
    assert sel(ms, batch=1) == 1 and sel(ms, batch=2) == 2 and sel(ms, batch=2, trip=2) == 3
    assert sel(ms, workgroup=512) == 0 and sel(ms, workgroup=1024, batch=1) == 1
    assert sel(ms, trip=8) == 5        # a trip narrows the batched candidates only
    assert sel(ms, batch=4) == 0       # no FP64 kernel has four nodes
    assert sel(ms, av=[1, 1, 1, 1, 0, 0], batch=0) == 0
    assert sq.tune_select(sq.SQ_FP32, [1] * 6, [5.0, 4.0, 3.0, 6.0, 2.0, 1.0], batch=0) == 0
    assert sq.tune_select(sq.SQ_FP32, [1] * 6, [5.0, 4.0, 3.0, 6.0, 2.0, 1.0], batch=4) == 5


def _run(monkeypatch, **env):
    for k in KERNEL_ENV + ("SQ_NO_RESIDENT",):
        monkeypatch.delenv(k, raising=False)
    for k, v in env.items():
        monkeypatch.setenv(k, v)
    with sq.Context(MG1, "Mg1", phantom_atom=True) as c:
        c.run(sq.SQ_NL_KB, sq.SQ_FP64, begin=1001, count=33)
        I = c.info
        return c.lanczos(), c.resident_planes(), (I.batch[0], I.workgroup[0], I.gather_trip[0])


@pytest.mark.gpu
@pytest.mark.parametrize("pins,kernel", [({"SQ_BATCH": "1", "SQ_ZMARCH_WG": "512"}, (1, 512, 0)),
                                         ({"SQ_ZMARCH_WG": "1024"}, (1, 1024, 0)),
                                         ({"SQ_BATCH": "2", "SQ_BATCH_TRIP": "1"}, (2, 1024, 1)),
                                         ({"SQ_BATCH": "2", "SQ_BATCH_TRIP": "2"}, (2, 1024, 2)),
                                         ({"SQ_BATCH": "4"}, (1, 512, 0))])
def test_pinned_column_marching_kernels_run(monkeypatch, pins, kernel):
    ab, planes, info = _run(monkeypatch, **pins)
    ref, none, info_ref = _run(monkeypatch, SQ_NO_RESIDENT="1", **pins)
    assert planes == 0 and none == 0 and info == kernel and info_ref == kernel
    assert np.array_equal(ab[0], ref[0]) and np.array_equal(ab[1], ref[1])


@pytest.mark.gpu
def test_resident_kernel_by_default_and_by_name(monkeypatch):
    ab, planes, info = _run(monkeypatch)
    named, planes_named, info_named = _run(monkeypatch, SQ_BATCH="0")
    assert planes > 0 and planes_named == planes and info == info_named == (0, 512, 0)   # 21^3: 441 columns
    assert np.array_equal(ab[0], named[0]) and np.array_equal(ab[1], named[1])


@pytest.mark.gpu
@pytest.mark.parametrize("wg", ["512", "1024"])
def test_one_node_kernel_stops_early_as_a_shorter_run(monkeypatch, tmp_path, wg):
    """FP64 in the pinned one-node kernel: a node that stops equals a fixed run of its length."""
    deck = write_variant(str(tmp_path), "L", nqp=40)
    for k in KERNEL_ENV + ("SQ_NO_RESIDENT",):
        monkeypatch.delenv(k, raising=False)
    monkeypatch.setenv("SQ_ZMARCH_WG", wg)
    with sq.Context(*deck) as c:
        assert c.resident_planes() == 0 and c.info.batch[0] == 1 and c.info.workgroup[0] == int(wg)
        c.run(sq.SQ_NL_KB, sq.SQ_FP64)
        lf = c.density_fermi_energy()[0]
        c.set_early_exit(1e-3, lf, 0.0, 12, 4)
        c.run(sq.SQ_NL_KB, sq.SQ_FP64)
        lam, w, _, _ = c.results()
        sizes = c.rule_sizes()
    assert sizes.min() >= 12 and np.any(sizes < 40)
    for s in sorted(set(sizes.tolist()))[:2]:
        with sq.Context(*deck, nqp=int(s)) as cs:
            for i in np.nonzero(sizes == s)[0][:3]:
                cs.run(sq.SQ_NL_KB, sq.SQ_FP64, begin=int(i), count=1)
                ls, ws, _, _ = cs.results()
                assert np.array_equal(lam[i, :s], ls[0]) and np.array_equal(w[i, :s], ws[0]), (i, s)
                assert np.all(w[i, s:] == 0.0)
