"""The kernels a plan's templates take, by steps, starts and flags, and the
autotuner's keys for them."""

import numpy as np
import pytest

from pyfstat_amd import _hiplib, autotune, synth
from pyfstat_amd.atoms import (
    TRANSIENT_EXPONENTIAL,
    TRANSIENT_RECTANGULAR,
    transientWindowRange_t,
)
from tests.test_gpu_rect_blocks import _atoms

pytestmark = pytest.mark.gpu

TA = synth.TSFT
RECT, EXP = TRANSIENT_RECTANGULAR, TRANSIENT_EXPONENTIAL
# (window type, N_t0, N_tau, t0 offset from the data's start, dt0, tau, dtau, generic): kernel
DISPATCH = [
    ((RECT, 20, 30, 0, TA, 2 * TA, TA, False), "rect_fast"),
    ((RECT, 20, 30, 77, 3 * TA, 5, 3 * TA, False), "rect_fast"),
    ((RECT, 20, 30, 0, TA, 2 * TA, 2 * TA, False), "rect_step"),
    ((RECT, 20, 30, -899, TA + 1, 2 * TA, TA + 700, False), "rect_step"),
    ((RECT, 1, 30, 0, 7, 2 * TA, TA + 1, False), "rect_step"),
    ((RECT, 20, 1, 0, TA + 1, 2 * TA, 7, False), "rect_step"),
    ((RECT, 20, 30, 0, TA - 1, 2 * TA, TA, False), "rect_generic"),
    ((RECT, 20, 30, 0, TA, 2 * TA, TA - 1, False), "rect_generic"),
    ((RECT, 20, 30, -901, TA, 2 * TA, TA, False), "rect_generic"),
    ((RECT, 20, 30, 0, TA, 2 * TA, TA, True), "rect_generic"),
    ((EXP, 20, 30, 0, TA, 2 * TA, TA, False), "exp_fast"),
    ((EXP, 20, 30, 1, TA, 2 * TA, TA, False), "exp_walk"),
    ((EXP, 20, 30, 0, TA + 1, 2 * TA, 5, False), "exp_walk"),
    ((EXP, 1, 30, 0, 7, 2 * TA, TA + 1, False), "exp_walk"),
    ((EXP, 20, 30, 0, TA - 1, 2 * TA, TA, False), "exp_direct"),
    ((EXP, 20, 30, 0, TA, TA - 1, TA, False), "exp_direct"),
    ((EXP, 20, 30, -1, TA, 2 * TA, TA, False), "exp_direct"),
    ((EXP, 20, 30, 0, TA, 2 * TA, TA, True), "exp_direct"),
]


def _batch(cases, ts, cols):
    from pyfstat_amd.batched import BatchedTransientMaps

    T = len(cases)
    wins = [transientWindowRange_t(type=kind, t0=int(ts[0]) + o, t0Band=(nt0 - 1) * dt0, dt0=dt0,
                                   tau=tau, tauBand=(ntau - 1) * dtau, dtau=dtau)
            for kind, nt0, ntau, o, dt0, tau, dtau, _ in cases]
    off = np.arange(T + 1, dtype=np.int64) * ts.size
    return BatchedTransientMaps(np.tile(ts, T), np.tile(cols, (1, T)), off,
                                np.arange(T + 1, dtype=np.int64), wins, TA, BtSG=True,
                                force_generic=cases[0][-1])


def test_kernels_by_steps_starts_and_flags(hip_ready):
    ts, cols = _atoms(200, 3, "plain")
    for case, kernel in DISPATCH:
        b = _batch([case], ts, cols)
        assert b.templates_per_kernel() == {k: int(k == kernel) for k in _hiplib.KERNEL_MODES}
        assert b.items_per_mode()[_hiplib.KERNEL_MODES[kernel]] > 0
        b.close()
    cases = [c for c, _ in DISPATCH if not c[-1]]
    b = _batch(cases, ts, cols)
    names = [k for c, k in DISPATCH if not c[-1]]
    assert b.templates_per_kernel() == {k: names.count(k) for k in _hiplib.KERNEL_MODES}
    b.close()


def test_keys_tell_the_kernels_of_a_mode_apart(hip_ready):
    ts, cols = _atoms(200, 3, "plain")
    for mode, names in ((_hiplib.MODE_RECT_GENERIC, ("rect_step", "rect_generic")),
                        (_hiplib.MODE_EXP_DIRECT, ("exp_walk", "exp_direct"))):
        keys = set()
        for name in names:
            b = _batch([next(c for c, k in DISPATCH if k == name)], ts, cols)
            keys.add(autotune.shape_class(b, mode, "dev"))
            b.close()
        assert len(keys) == 2
