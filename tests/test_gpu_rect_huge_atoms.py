"""The regular-grid rect kernel where determinants leave the float32 range: the
condition test of a lane's cells at once against the generic kernel's cell by
cell, and the maximum's position inside the map."""

import numpy as np
import pytest

from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR
from tests.test_gpu_rect_blocks import _atoms

pytestmark = pytest.mark.gpu

N_TAUS = (1, 64, 256, 257, 300, 385, 512)


def _batch(kind, n_t0, generic):
    from pyfstat_amd.batched import BatchedTransientMaps

    # (tiny: all windows past the first column block end with the data, and a
    # wave's lanes agree)
    ts, cols = _atoms(250 if kind == "tiny" else 700, 7, "plain")
    cols = cols.astype(np.float64)
    cols[:3] *= 1e24  # determinants of 1e48 and more
    if kind == "degenerate":  # condition numbers near 4e5: F = 2 in every cell
        cols[1] = cols[0]
        cols[2] = cols[0] * (1.0 - 5e-6)
    elif kind == "tiny":  # determinants of a few units of the last float32 place there is
        cols[:3] *= 2e-46
        cols[1] = cols[0]
        cols[2] = cols[0] * np.sqrt(1.0 - 4.0 / (1.0003 * 10001.0**2 / 1e4))
    elif kind == "some":  # until some way into the data
        k = cols.shape[1] // 2
        cols[1, :k] = cols[0, :k]
        cols[2, :k] = cols[0, :k] * (1.0 - 5e-6)
        cols[:3, k:] *= 1e-3
    cols = cols.astype(np.float32)
    T = len(N_TAUS)
    wins = [synth.grid_window(TRANSIENT_RECTANGULAR, synth.T_START, n_t0, k) for k in N_TAUS]
    off = np.arange(T + 1, dtype=np.int64) * ts.size
    return BatchedTransientMaps(np.tile(ts, T), np.tile(cols, (1, T)), off,
                                np.arange(T + 1, dtype=np.int64), wins, synth.TSFT, BtSG=True,
                                force_generic=generic)


@pytest.mark.parametrize("kind", ["plain", "degenerate", "some", "tiny"])
@pytest.mark.parametrize("n_t0", [1, 3, 17, 200])
def test_determinants_out_of_range_match_generic_kernel(hip_ready, kind, n_t0):
    fast, ref = _batch(kind, n_t0, False), _batch(kind, n_t0, True)
    assert fast.items_per_mode()[0] > 0 and ref.items_per_mode()[1] > 0
    fast.run()
    ref.run()
    F, G = fast.F_host(), ref.F_host()
    np.testing.assert_array_equal(F, G)
    if kind == "degenerate":
        assert np.all(G == 2.0)
    st, sg = fast.stats(), ref.stats()
    for f in ("maxF", "m_ML", "n_ML"):
        np.testing.assert_array_equal(st[f], sg[f])
    assert np.all(st["m_ML"] < n_t0) and np.all(st["n_ML"] < np.array(N_TAUS))
    fast.close()
    ref.close()
