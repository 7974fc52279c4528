"""Regular rectangular grids whose steps are so many atoms that the start index of
a row past the map does not fit 32 bits: they go to the step kernel, and their
maps match the oracle's."""

import numpy as np
import pytest

import oracle
from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR, transientWindowRange_t
from tests.helpers import compare_maps

pytestmark = pytest.mark.gpu

TA = 2
T0 = 1_000_000_000
WIDEST = 2**32 - 2


@pytest.mark.parametrize("n_t0,n_tau,step,kernel", [
    (1, 1, WIDEST, "rect_step"),        # 3 steps past the map overflow
    (2, 1, 2**31 - 2, "rect_step"),
    (1, 2, 2**31 - 2, "rect_step"),
    (1, 1, 2**30, "rect_fast"),         # 3 * 2^29 still fit
    (3, 2, 2**28, "rect_fast"),
])
def test_steps_of_billions_of_atoms(hip_ready, n_t0, n_tau, step, kernel):
    from pyfstat_amd.batched import BatchedTransientMaps

    rng = np.random.default_rng(5)
    t = (T0 + TA * np.arange(300)).astype(np.uint32)
    cols = synth.detector_atoms(rng, t.astype(float), 0.3, 1.1, np.zeros(t.size, complex))
    win = transientWindowRange_t(type=TRANSIENT_RECTANGULAR, t0=T0, t0Band=(n_t0 - 1) * step,
                                 dt0=step, tau=400, tauBand=(n_tau - 1) * step, dtau=step)
    assert T0 + win.t0Band + win.tau + win.tauBand + 1 < 2**32
    b = BatchedTransientMaps(t, cols, np.array([0, t.size]), np.array([0, 1]), [win], TA,
                             BtSG=True)
    assert b.templates_per_kernel()[kernel] == 1
    b.run()
    merged, t_min = oracle.merge_binned(t, cols, np.array([0, t.size]), TA)
    om = oracle.compute_map(merged, TA, t_min, win)
    m = b.maps()[0]
    compare_maps(m.F_mn, om)
    assert tuple(int(i) for i in m.get_maxF_idx()) == (om.m_max, om.n_max)
    b.close()
