"""tcw_map_noalloc at the edge of the static scratch: what it accepts is decided
by one layout (16 rows x 256 columns an item off the atom grid, chunks of 64 rows
on it), whichever layout then runs."""

import ctypes

import numpy as np
import pytest

from pyfstat_amd import _hiplib, synth
from pyfstat_amd.atoms import TRANSIENT_EXPONENTIAL, transientWindowRange_t
from tests.test_zz_no_alloc import _both

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("n_tau,compact", [(8_000_000, True), (1_000_000, False)])
def test_wide_map_off_the_grid_fits(hip_ready, n_tau, compact):
    # per column 4 bytes of column partials, per item 4 of row partials, 16 of
    # descriptor and 16 of results
    def need(tile):
        return 4 * n_tau + 36 * -(-n_tau // tile)

    assert need(256) < _hiplib.TCW_NOALLOC_SCRATCH_BYTES - 65536
    assert (need(64) > _hiplib.TCW_NOALLOC_SCRATCH_BYTES) == compact
    multi, _ = synth.workload_exp_plain(n_sft=90, n_t0=10, n_tau=10, seed_index=77)
    win = transientWindowRange_t(type=TRANSIENT_EXPONENTIAL, t0=synth.T_START, t0Band=0, dt0=100,
                                 tau=2 * synth.TSFT, tauBand=n_tau - 1, dtau=1)
    F_ref, st_ref, F, st = _both(multi, win, _hiplib.TCW_FLAG_BTSG)
    assert F.shape == (1, n_tau)
    # FP64 sums of 90 terms, 1e-14 apart, times the condition number (< 1e4),
    # and the float32 quotient (3e-7 on either side)
    np.testing.assert_allclose(F, F_ref, rtol=1e-6, atol=1e-7)
    assert st.maxF == F.max() and int(st.n_ML) == int(F.argmax()) and int(st.m_ML) == 0
    assert abs(st.lnBtSG - st_ref.lnBtSG) <= 2e-6 + 6e-7 * abs(st.maxF)
    if not compact:
        np.testing.assert_array_equal(F, F_ref)


def test_map_at_the_end_of_long_data_fits(hip_ready):
    # the atom table of all bins leaves room for the E tables of chunks of 64
    # rows (37 + 2 + 8 slots of 7 doubles a column), not of 32 (over 80)
    N, n_t0, n_tau = 935_000, 100, 1000
    room = _hiplib.TCW_NOALLOC_SCRATCH_BYTES - 32 * N
    assert 50 * 56 * n_tau + 65536 < room < 80 * 56 * n_tau
    rng = np.random.default_rng(78)
    idx = np.concatenate([[0], np.arange(N - 2500, N)])
    t = synth.T_START + idx * float(synth.TSFT)
    cols = synth.detector_atoms(rng, t, 0.4, 1.2, np.zeros(t.size, complex))
    multi = synth.multi_from_detectors([(t.astype(np.uint32), cols)])
    win = synth.grid_window(TRANSIENT_EXPONENTIAL, synth.T_START + (N - 2400) * synth.TSFT, n_t0,
                            n_tau)
    F_ref, st_ref, F, st = _both(multi, win, _hiplib.TCW_FLAG_BTSG)
    assert F.shape == (n_t0, n_tau)
    # FP64 sums of 2400 terms, 1e-13 apart, times the condition number (< 1e4
    # and below 10 but for the shortest windows), and the float32 quotient
    np.testing.assert_allclose(F, F_ref, rtol=1e-6, atol=1e-7)
    assert st.maxF == F.max() and abs(st.lnBtSG - st_ref.lnBtSG) <= 2e-6 + 6e-7 * st.maxF


def test_map_that_only_a_shorter_layout_holds_is_refused(hip_ready):
    import torch

    from pyfstat_amd import tcw_fstat_map_funcs as tcw
    from tests.test_zz_no_alloc import _device_atoms

    n_t0, n_tau = 256, 600_000
    # column partials of items of 16 rows, of 256 rows
    assert n_t0 // 16 * n_tau * 4 > _hiplib.TCW_NOALLOC_SCRATCH_BYTES > 4 * n_tau * 4
    lib = _hiplib.load()
    handle = tcw._ensure_handle()
    dev = torch.device("cuda", tcw._HipState.device)
    multi, _ = synth.workload_exp_plain(n_sft=600, n_t0=10, n_tau=10, seed_index=79)
    packed, at, keep = _device_atoms(multi, dev)
    win = _hiplib.Window(type=TRANSIENT_EXPONENTIAL, t0=synth.T_START, t0Band=(n_t0 - 1) * 900,
                         dt0=900, tau=2 * synth.TSFT, tauBand=n_tau - 1, dtau=1)
    F = torch.zeros(n_t0, n_tau, dtype=torch.float32, device=dev)
    st = torch.empty(_hiplib.STATS_BYTES, dtype=torch.uint8, device=dev)
    rc = lib.tcw_map_noalloc(handle, ctypes.byref(at), ctypes.byref(win),
                             ctypes.c_void_p(F.data_ptr()), ctypes.c_void_p(st.data_ptr()),
                             _hiplib.TCW_FLAG_BTSG,
                             ctypes.c_void_p(torch.cuda.current_stream(dev).cuda_stream))
    assert rc == _hiplib.TCW_ERR_INVALID
    assert b"static scratch holds" in lib.tcw_last_error()
    torch.cuda.synchronize()
    assert not F.any()
    del keep
