"""Rectangular windows whose start and duration steps are both an atom or more
and neither a whole number of atoms: the step kernel, which takes them, against
the generic per-cell kernel (the same prefix table, window indices and cell
formula, so every bit is the same).  Steps below one atom, which the generic
kernel takes, against the FP64 oracle."""

import numpy as np
import pytest

import oracle
from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR, transientWindowRange_t
from tests.helpers import check_argmax, compare_maps
from tests.test_gpu_parity import _posterior_ok, lnb_tol
from tests.test_gpu_rect_blocks import _atoms

TA = synth.TSFT
N_BINS = 3000
# (N_t0, N_tau, t0 offset from the data's start, dt0, tau, dtau): one to four
# column groups and several blocks; starts before, within and a bin after the
# data's first; durations just below a whole number of bins; the last two have
# ranges too wide for LDS at any width
GRIDS = [
    (64, 64, 899, TA + 1, 3 * TA - 1, TA + 1),
    (33, 65, -899, TA + 700, 2 * TA - 1, TA + 1799),
    (130, 129, 1000, 2 * TA - 1, 5399, 2 * TA - 1),
    (70, 257, 773, TA + 974, 2 * TA, TA + 362),
    (21, 300, 800, 3 * TA + 11, TA + 1797, TA + 5),
    (17, 520, -900, 2 * TA + 901, 0, 3 * TA + 899),
    (200, 40, 450, 7 * TA + 599, 10 * TA + 1201, 5 * TA + 1),
    (50, 90, 835, 20 * TA + 7, 2 * TA, 30 * TA + 1799),
    (40, 300, 899, 2 * TA + 1, TA, 25 * TA + 1),
]
SUB_ATOM = [
    (20, 300, 899, 901, 1, 700),
    (64, 65, -899, 1799, TA, 1801),
    (50, 129, 0, 7, 2 * TA, 8 * TA),
    (48, 600, 13, 123, 2 * TA, 11 * TA),
    (37, 30, 5, 5 * TA, 2 * TA - 1, 450),
]


def _windows(grids, t_min):
    return [transientWindowRange_t(type=TRANSIENT_RECTANGULAR, t0=t_min + o,
                                   t0Band=(nt0 - 1) * dt0, dt0=dt0, tau=tau,
                                   tauBand=(ntau - 1) * dtau, dtau=dtau)
            for nt0, ntau, o, dt0, tau, dtau in grids]


def _batch(grids, kind, generic, rows=None):
    from pyfstat_amd.batched import BatchedTransientMaps

    ts, cols = _atoms(N_BINS, 17, kind)
    T = len(grids)
    off = np.arange(T + 1, dtype=np.int64) * ts.size
    return BatchedTransientMaps(np.tile(ts, T), np.tile(cols, (1, T)), off,
                                np.arange(T + 1, dtype=np.int64), _windows(grids, int(ts[0])), TA,
                                BtSG=True, force_generic=generic,
                                rows=None if rows is None else {1: rows})


def test_grids_reach_what_they_are_for():
    """On the CPU: the rule that sends a grid to the step kernel, and carries of
    the end's remainder and wraps of the start's, in every column count."""
    early = 0
    for nt0, ntau, o, dt0, tau, dtau in GRIDS:
        assert dt0 >= TA and dtau >= TA and dt0 % TA and dtau % TA
        assert o + TA // 2 >= 0
        early += o < 0
        T = o + TA // 2 + np.arange(nt0) * dt0
        x = tau + np.arange(ntau) * dtau
        carry = (T % TA)[:, None] + (x % TA)[None, :] >= TA
        assert carry.any() and not carry.all()
        wrap = (T[:-1] % TA) + dt0 % TA >= TA
        wrap[3::4] = False  # within the four rows of a wave
        assert wrap.any()
    assert early >= 2
    for nt0, ntau, o, dt0, tau, dtau in SUB_ATOM:
        assert dt0 < TA or dtau < TA


@pytest.mark.gpu
@pytest.mark.parametrize("kind", ["plain", "nan"])
@pytest.mark.parametrize("rows", [None, 16, 128])
def test_fractional_steps_match_generic_kernel(hip_ready, kind, rows):
    b, ref = _batch(GRIDS, kind, False, rows), _batch(GRIDS, kind, True)
    assert b.items_per_mode()[1] > 0 and b.items_per_mode()[0] == 0
    b.run()
    ref.run()
    np.testing.assert_array_equal(b.F_host(), ref.F_host())
    st, sg = b.stats(), ref.stats()
    for f in ("maxF", "m_ML", "n_ML"):
        np.testing.assert_array_equal(st[f], sg[f])
    if kind == "plain":
        # the same float32 terms in other orders: 1e-6 of a sum of at most 1e5 terms
        np.testing.assert_allclose(st["lnBtSG"], sg["lnBtSG"], rtol=0, atol=2e-6)
    b.close()
    ref.close()


@pytest.mark.gpu
@pytest.mark.parametrize("grids", [GRIDS, SUB_ATOM], ids=["atom", "sub_atom"])
def test_fractional_steps_match_oracle(hip_ready, grids):
    ts, cols = _atoms(N_BINS, 17, "plain")
    merged, t0 = oracle.merge_binned(ts, cols, np.array([0, ts.size]), TA)
    b = _batch(grids, "plain", False)
    b.run()
    for m, win in zip(b.maps(), b.windows):
        om = oracle.compute_map(merged, TA, t0, win)
        om.lnBtSG = oracle.lnBtSG(om.F_mn, om.maxF)
        compare_maps(m.F_mn, om)
        check_argmax(m.F_mn, *(int(i) for i in m.get_maxF_idx()), om)
        assert abs(m.lnBtSG - om.lnBtSG) <= lnb_tol(om.maxF)
        _posterior_ok(om, win, m.t0_MP, m.tau_MP)
    b.close()
