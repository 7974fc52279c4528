"""The regular-grid rect kernel's column layouts, condition test and position
of the maximum, at the sizes where they change, against the generic per-cell
kernel (the same prefix table and cell formula, so every bit is the same)."""

import numpy as np
import pytest

from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR

pytestmark = pytest.mark.gpu

N_TAUS = (1, 2, 3, 4, 63, 64, 65, 127, 128, 129, 255, 256, 257, 320, 321, 384, 385, 512)


def _atoms(n, seed, kind):
    rng = np.random.default_rng(seed)
    idx = np.nonzero(synth.gap_mask(rng, n, 0.1))[0]
    t = synth.T_START + idx * float(synth.TSFT)
    cols = synth.detector_atoms(rng, t, 0.3, 1.1, np.zeros(t.size, complex))
    k = t.size
    if kind == "negative":  # traces that do not grow with the window
        cols[0, k // 3] = -5.0
        cols[1, k // 2] = -5.0
    elif kind == "indefinite":  # determinants of either sign at short and long windows
        cols[2] *= 3.0
    elif kind == "nan":
        cols[2, k // 2] = np.nan
    elif kind == "inf":
        cols[0, k // 2] = np.inf
    elif kind == "zero":  # every window degenerate: F = 2 everywhere
        cols[:] = 0.0
    elif kind == "aligned":  # one antenna direction: determinants of rounding size
        cols[1] = cols[0]
        cols[2] = cols[0]
    return t.astype(np.uint32), cols


def _batch(kind, n_t0, btsg, generic, rows=None, step=1, n=700):
    from pyfstat_amd.batched import BatchedTransientMaps

    ts, cols = _atoms(n, 7, kind)
    T = len(N_TAUS)
    wins = [synth.grid_window(TRANSIENT_RECTANGULAR, synth.T_START, n_t0, k, dt0=step * synth.TSFT,
                              dtau=step * synth.TSFT) for k in N_TAUS]
    off = np.arange(T + 1, dtype=np.int64) * ts.size
    return BatchedTransientMaps(np.tile(ts, T), np.tile(cols, (1, T)), off,
                                np.arange(T + 1, dtype=np.int64), wins, synth.TSFT, BtSG=btsg,
                                force_generic=generic, rows=None if rows is None else {0: rows})


@pytest.mark.parametrize("kind", ["plain", "negative", "indefinite", "nan", "inf", "zero",
                                  "aligned"])
@pytest.mark.parametrize("n_t0,btsg,rows,step", [(1, True, None, 1), (3, False, None, 1),
                                                 (17, True, 16, 1), (200, True, None, 1),
                                                 (200, True, 192, 3), (333, False, 512, 1)])
def test_layouts_match_generic_kernel(hip_ready, kind, n_t0, btsg, rows, step):
    fast = _batch(kind, n_t0, btsg, False, rows, step)
    ref = _batch(kind, n_t0, btsg, True, None, step)
    assert fast.items_per_mode()[0] > 0 and ref.items_per_mode()[1] > 0
    fast.run()
    ref.run()
    F, G = fast.F_host(), ref.F_host()
    np.testing.assert_array_equal(F, G)
    st, sg = fast.stats(), ref.stats()
    for t in range(fast.T):
        m = fast.map_view(F, t)
        if np.isnan(m).all():
            continue
        first = int(np.nanargmax(m))  # first row-major occurrence
        assert st["maxF"][t] == m.reshape(-1)[first]
        assert (int(st["m_ML"][t]), int(st["n_ML"][t])) == divmod(first, m.shape[1])
    if btsg and kind not in ("nan", "inf", "negative", "indefinite"):
        # both kernels sum the same float32 terms in other orders: 1e-6 of a
        # sum of at most 1e5 terms
        np.testing.assert_allclose(st["lnBtSG"], sg["lnBtSG"], rtol=0, atol=2e-6)
    fast.close()
    ref.close()
