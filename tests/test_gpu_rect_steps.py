"""Rectangular windows with start and duration steps of any size: the step
kernel against the generic per-cell kernel (the same prefix table, window
indices and cell formula, so every bit is the same)."""

import numpy as np
import pytest

from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR, transientWindowRange_t
from tests.test_gpu_rect_blocks import _atoms

pytestmark = pytest.mark.gpu

TA = synth.TSFT
# (N_t0, N_tau, t0 offset, dt0, tau, dtau): steps of part of a bin, odd and even
# numbers of bins, ranges too wide for LDS, starts before the data (by less
# than half a bin), windows of no bin, and starts and ends past the data
GRIDS = [
    (1, 1, 0, 1, 0, 1),
    (5, 255, 0, TA, 2 * TA, 2 * TA),
    (17, 256, 0, 2 * TA, 2 * TA, 3 * TA),
    (33, 257, 450, 3 * TA, 2 * TA, 2 * TA),
    (20, 300, 899, 901, 1, 700),
    (64, 65, -899, 1799, TA, 1801),
    (16, 520, 0, TA, 2 * TA, 4 * TA),
    (50, 129, 0, 7, 2 * TA, 8 * TA),
    (19, 300, 77, 40 * TA + 11, 3, 6 * TA),
    (90, 40, 0, 5 * TA, 30 * TA, 60 * TA + 1),
    (48, 600, 13, 123, 2 * TA, 11 * TA),
]


def _batch(kind, generic, btsg, rows=None):
    from pyfstat_amd.batched import BatchedTransientMaps

    ts, cols = _atoms(700, 11, kind)
    T = len(GRIDS)
    wins = [transientWindowRange_t(type=TRANSIENT_RECTANGULAR, t0=synth.T_START + o,
                                   t0Band=(nt0 - 1) * dt0, dt0=dt0, tau=tau,
                                   tauBand=(ntau - 1) * dtau, dtau=dtau)
            for nt0, ntau, o, dt0, tau, dtau in GRIDS]
    off = np.arange(T + 1, dtype=np.int64) * ts.size
    return BatchedTransientMaps(np.tile(ts, T), np.tile(cols, (1, T)), off,
                                np.arange(T + 1, dtype=np.int64), wins, TA, BtSG=btsg,
                                force_generic=generic, rows=None if rows is None else {1: rows})


@pytest.mark.parametrize("kind", ["plain", "negative", "nan", "zero"])
@pytest.mark.parametrize("btsg,rows", [(True, None), (False, 16), (True, 64)])
def test_steps_match_generic_kernel(hip_ready, kind, btsg, rows):
    b, ref = _batch(kind, False, btsg, rows), _batch(kind, True, btsg)
    assert b.items_per_mode()[0] == 0 and b.items_per_mode()[1] > 0
    for x in (b, ref):
        x.flags |= 2  # single-atom windows too
        x.replan()
        x.run()
    F, G = b.F_host(), ref.F_host()
    np.testing.assert_array_equal(F, G)
    st, sg = (x.stats_d.cpu().numpy().view(_stats()) for x in (b, ref))
    for f in ("maxF", "m_ML", "n_ML", "single_atom"):
        np.testing.assert_array_equal(st[f], sg[f])
    if btsg and kind in ("plain", "zero"):
        # the same float32 terms in other orders: 1e-6 of a sum of at most 1e5 terms
        np.testing.assert_allclose(st["lnBtSG"], sg["lnBtSG"], rtol=0, atol=2e-6)
    b.close()
    ref.close()


def _stats():
    from pyfstat_amd.batched import STATS_DTYPE

    return STATS_DTYPE
