"""Exponential windows with starts an atom or more apart at every phase: the
sliding sum, which takes them, against the direct sum of every cell.  Starts less
than an atom apart, which keep the direct sum, against the FP64 oracle."""

import numpy as np
import pytest

import oracle
from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_EXPONENTIAL, transientWindowRange_t
from tests.helpers import check_argmax, compare_maps
from tests.test_gpu_exp_walk_steps import _atoms
from tests.test_gpu_parity import _posterior_ok, lnb_tol

pytestmark = pytest.mark.gpu

TA = synth.TSFT
# (N_t0, N_tau, t0 offset from the data's start, dt0, tau, dtau): one to five
# column groups, starts and ends of every phase, duration steps of part of an
# atom to many, starts longer apart than the shortest windows, and past the data
GRIDS = [
    (5, 63, 0, TA + 900, 2 * TA, 900),
    (17, 64, 7, TA + 601, 2 * TA, 2700),
    (64, 200, 1799, 2 * TA - 1, 2 * TA + 1, 4500),
    (35, 300, 13, TA + 1000, 5 * TA, 40 * TA + 11),
    (130, 65, 901, TA, TA + 1, 1),
    (257, 33, 1, TA + 1, 3 * TA + 7, 450),
    (90, 129, 900, 3 * TA + 1799, TA, TA - 1),
    (40, 100, 450, 9 * TA + 3, TA + 5, 700),
]
SUB_ATOM = [
    (5, 63, 0, 900, 2 * TA, 900),
    (17, 64, 7, 601, 2 * TA, 2700),
    (64, 200, 1799, 1799, 2 * TA + 1, 4500),
    (35, 300, 13, 1000, 5 * TA, 40 * TA + 11),
    (100, 23, 0, TA // 2, 2 * TA, 4500),
    (100, 23, 0, TA // 4, 2 * TA, 4500),
]


def _data(k, kind, n_det):
    dets = _atoms(400, 80 + k, kind, n_det)
    return dets, min(int(t[0]) for t, _ in dets)


def _batch(grids, kind, n_det, generic, rows=None):
    from pyfstat_amd.batched import BatchedTransientMaps

    ts, cols, off, begin, wins = [], [], [0], [0], []
    for k, (nt0, ntau, o, dt0, tau, dtau) in enumerate(grids):
        dets, t_min = _data(k, kind, n_det)
        for t, c in dets:
            ts.append(t)
            cols.append(c)
            off.append(off[-1] + t.size)
        begin.append(len(off) - 1)
        wins.append(transientWindowRange_t(
            type=TRANSIENT_EXPONENTIAL, t0=t_min + o, t0Band=(nt0 - 1) * dt0, dt0=dt0, tau=tau,
            tauBand=(ntau - 1) * dtau, dtau=dtau))
    return BatchedTransientMaps(np.concatenate(ts), np.concatenate(cols, 1), off, begin, wins, TA,
                                BtSG=True, force_generic=generic,
                                rows=None if rows is None else {2: rows})


@pytest.mark.parametrize("kind", ["plain", "gap"])
@pytest.mark.parametrize("n_det,rows", [(1, None), (2, 16), (2, 64), (1, 512)])
def test_sliding_sum_matches_direct_sum(hip_ready, kind, n_det, rows):
    b, ref = _batch(GRIDS, kind, n_det, False, rows), _batch(GRIDS, kind, n_det, True)
    assert b.templates_per_kernel()["exp_walk"] == b.T
    assert ref.templates_per_kernel()["exp_direct"] == b.T
    b.run()
    ref.run()
    F, G = b.F_host(), ref.F_host()
    st, sg = b.stats(), ref.stats()
    # FP64 sums of a few hundred terms, 1e-13 apart, times the condition
    # number (< 1e4), then the float32 quotient (3e-7 on either side)
    np.testing.assert_allclose(F, G, rtol=1e-6, atol=1e-7)
    assert np.array_equal(F == 2.0, G == 2.0)
    for t in range(b.T):
        m = b.map_view(F, t)
        first = int(m.argmax())
        assert st["maxF"][t] == m.reshape(-1)[first]
        assert (int(st["m_ML"][t]), int(st["n_ML"][t])) == divmod(first, m.shape[1])
        # 1e-6 of the sum, and F's rounding times F
        assert abs(st["lnBtSG"][t] - sg["lnBtSG"][t]) <= 2e-6 + 6e-7 * abs(st["maxF"][t])
    b.close()
    ref.close()


@pytest.mark.parametrize("grids,kernel", [(GRIDS, "exp_walk"), (SUB_ATOM, "exp_direct")],
                         ids=["atom", "sub_atom"])
def test_maps_match_oracle(hip_ready, grids, kernel):
    b = _batch(grids, "plain", 2, False)
    assert b.templates_per_kernel()[kernel] == b.T
    b.run()
    for k, (m, win) in enumerate(zip(b.maps(), b.windows)):
        dets, t_min = _data(k, "plain", 2)
        off = np.cumsum([0] + [t.size for t, _ in dets])
        merged, t0 = oracle.merge_binned(np.concatenate([t for t, _ in dets]),
                                         np.concatenate([c for _, c in dets], 1), off, TA)
        assert t0 == t_min
        om = oracle.compute_map(merged, TA, t0, win)
        om.lnBtSG = oracle.lnBtSG(om.F_mn, om.maxF)
        compare_maps(m.F_mn, om)
        check_argmax(m.F_mn, *(int(i) for i in m.get_maxF_idx()), om)
        assert abs(m.lnBtSG - om.lnBtSG) <= lnb_tol(om.maxF)
        _posterior_ok(om, win, m.t0_MP, m.tau_MP)
    b.close()
