"""Exponential windows with steps off the atom grid: the sliding sum against
the direct sum of every cell (the generic path), where the sums agree to the
rounding of the stored float32, and with infinities and NaN in the data against
the FP64 oracle."""

import numpy as np
import pytest

import oracle
from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_EXPONENTIAL, transientWindowRange_t

pytestmark = pytest.mark.gpu

TA = synth.TSFT
# (N_t0, N_tau, t0 offset, dt0, tau, dtau): every phase of the start and end
# within an atom; one, two, three and four column groups; steps of part of an
# atom, many atoms, longer than the windows, and beyond the data
GRIDS = [
    (1, 1, 0, 1, TA, 1),
    (5, 63, 0, 900, 2 * TA, 900),
    (17, 64, 7, 601, 2 * TA, 2700),
    (40, 65, 901, 2700, TA, 450),
    (33, 130, 900, 2701, 3601, 1801),
    (64, 200, 1799, 1799, 2 * TA + 1, 4500),
    (30, 257, 0, 5400 + 1, 3600, 600),
    (12, 40, 450, 40 * TA + 450, 2 * TA, 300),
    (100, 30, 0, 8 * TA + 1, 30 * TA, 12 * TA + 7),
    (35, 300, 13, 1000, 5 * TA, 40 * TA + 11),
]


def _atoms(n, seed, kind, n_det):
    rng = np.random.default_rng(seed)
    dets = []
    for X in range(n_det):
        idx = np.nonzero(synth.gap_mask(rng, n, 0.1))[0]
        t = synth.T_START + idx * float(TA)
        cols = synth.detector_atoms(rng, t, 0.3 + X, 1.1 - X, np.zeros(t.size, complex))
        if kind == "gap":  # windows inside it hold no data at all
            cols[:, (idx > n // 4) & (idx < n // 2)] = 0.0
        elif kind == "nan":
            cols[3, t.size // 5] = np.nan
        elif kind == "inf":
            cols[0, t.size // 5] = np.inf
        dets.append((t.astype(np.uint32), cols))
    return dets


def _batch(kind, n_det, generic, rows, btsg=True, strict=False):
    from pyfstat_amd.batched import BatchedTransientMaps

    ts, cols, off, begin, wins = [], [], [0], [0], []
    for k, (nt0, ntau, o, dt0, tau, dtau) in enumerate(GRIDS):
        for t, c in _atoms(400, 40 + k, kind, n_det):
            ts.append(t)
            cols.append(c)
            off.append(off[-1] + t.size)
        begin.append(len(off) - 1)
        wins.append(transientWindowRange_t(
            type=TRANSIENT_EXPONENTIAL, t0=synth.T_START + o, t0Band=(nt0 - 1) * dt0, dt0=dt0,
            tau=tau, tauBand=(ntau - 1) * dtau, dtau=dtau))
    return BatchedTransientMaps(np.concatenate(ts), np.concatenate(cols, 1), off, begin, wins, TA,
                                BtSG=btsg, force_generic=generic,
                                rows=None if rows is None else {2: rows})


def _assert_argmax(b, F, st):
    for t in range(b.T):
        m = b.map_view(F, t)
        if np.isnan(m).all():
            continue
        first = int(np.nanargmax(m))
        assert st["maxF"][t] == m.reshape(-1)[first]
        assert (int(st["m_ML"][t]), int(st["n_ML"][t])) == divmod(first, m.shape[1])


@pytest.mark.parametrize("kind", ["plain", "gap"])
@pytest.mark.parametrize("n_det,rows", [(1, None), (2, 16), (2, 48), (1, 512)])
def test_sliding_sum_matches_direct_sum(hip_ready, kind, n_det, rows):
    b = _batch(kind, n_det, False, rows)
    ref = _batch(kind, n_det, True, None)
    assert b.items_per_mode()[2] > 0 and b.items_per_mode()[3] == 0
    b.run()
    ref.run()
    F, G = b.F_host(), ref.F_host()
    st, sg = b.stats(), ref.stats()
    # FP64 sums of a few hundred terms, 1e-13 apart, times the condition
    # number (< 1e4), then the float32 quotient (3e-7 on either side); a window
    # whose condition number lies within 1e-9 of the guard is not drawn here
    np.testing.assert_allclose(F, G, rtol=1e-6, atol=1e-7)
    assert np.array_equal(F == 2.0, G == 2.0)
    _assert_argmax(b, F, st)
    for t in range(b.T):
        # 1e-6 of the sum, and F's rounding times F
        assert abs(st["lnBtSG"][t] - sg["lnBtSG"][t]) <= 2e-6 + 6e-7 * abs(st["maxF"][t])
    b.close()
    ref.close()


@pytest.mark.parametrize("kind", ["nan", "inf"])
@pytest.mark.parametrize("rows", [None, 16, 128])
def test_infinite_and_nan_atoms_reach_their_windows_only(hip_ready, kind, rows):
    b = _batch(kind, 1, False, rows)
    b.run()
    F, st = b.F_host(), b.stats()
    for k in range(b.T):
        (ts, cols), = _atoms(400, 40 + k, kind, 1)
        merged, t0 = oracle.merge_binned(ts, cols, np.array([0, ts.size]), TA)
        om = oracle.compute_map(merged, TA, t0, b.windows[k])
        m = b.map_view(F, k)
        assert np.array_equal(np.isnan(m), np.isnan(om.F_mn))
        ok = ~np.isnan(m)
        np.testing.assert_allclose(m[ok], om.F_mn[ok], rtol=1e-6, atol=1e-7)
    _assert_argmax(b, F, st)
    b.close()


def test_single_atom_flag_matches_direct_sum(hip_ready):
    b = _batch("plain", 1, False, None, strict=True)
    ref = _batch("plain", 1, True, None, strict=True)
    for x in (b, ref):
        x.flags |= 2
        x.replan()
        x.run()
    import torch

    torch.cuda.synchronize()
    from pyfstat_amd.batched import STATS_DTYPE

    one, two = (x.stats_d.cpu().numpy().view(STATS_DTYPE)["single_atom"] for x in (b, ref))
    assert np.array_equal(one, two) and one.any() and not one.all()
    b.close()
    ref.close()


@pytest.mark.parametrize("dt0", [TA // 2, TA // 4, 700, TA + 1, 2700])
def test_equal_windows_keep_their_order(hip_ready, dt0):
    """Starts that step by part of an atom repeat windows, whose F are equal but for
    rounding: the maximum and the posterior's mode are the direct sum's, as are
    all but a few F of larger steps."""
    from pyfstat_amd.batched import BatchedTransientMaps

    maps = []
    for generic in (False, True):
        ts, cols, off, wins, T = [], [], [0], [], 24
        for k in range(T):
            (t, c), = _atoms(250, 300 + k, "plain", 1)
            ts.append(t)
            cols.append(c)
            off.append(off[-1] + t.size)
            wins.append(transientWindowRange_t(
                type=TRANSIENT_EXPONENTIAL, t0=synth.T_START, t0Band=99 * dt0, dt0=dt0,
                tau=2 * TA, tauBand=22 * 4500, dtau=4500))
        b = BatchedTransientMaps(np.concatenate(ts), np.concatenate(cols, 1), off,
                                 np.arange(T + 1), wins, TA, BtSG=True, force_generic=generic)
        b.run()
        maps.append((b.F_host(), b.stats()))
        b.close()
    (F, st), (G, sg) = maps
    # both round the same two FP64 numbers, 1e-13 apart, to float32: all but
    # about 1e-6 of the cells are the same float
    assert (F != G).mean() < 1e-4
    for f in ("m_ML", "n_ML", "m_MP", "n_MP"):
        np.testing.assert_array_equal(st[f], sg[f])
