"""What the autotuner times and how it keys what it keeps (host logic, no device)."""

import numpy as np
import pytest

from pyfstat_amd import _hiplib, autotune
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR, transientWindowRange_t

KERNELS = ("rect_fast", "rect_step", "rect_generic", "exp_direct", "exp_walk", "exp_fast")


class FakeBatch:
    T = 8
    TAtom = 1800

    def __init__(self, kernels, dt0=2700, dtau=2700):
        self.kernels = kernels  # templates of each kernel
        self.rows = {}
        self.windows = [transientWindowRange_t(type=TRANSIENT_RECTANGULAR, t0=0, t0Band=499 * dt0,
                                               dt0=dt0, tau=3600, tauBand=499 * dtau, dtau=dtau)
                        ] * self.T

    def _shape(self, t):
        return (500, 500)

    def templates_per_kernel(self):
        return {k: self.kernels.get(k, 0) for k in KERNELS}

    def items_per_mode(self):
        return np.ones(_hiplib.MODE_COUNT, dtype=np.int64)

    def set_rows(self, mode, rows):
        self.rows[int(mode)] = int(rows)

    @property
    def rows_by_mode(self):
        return [self.rows.get(m, 0) for m in range(_hiplib.MODE_COUNT)]

    def replan(self):
        pass


@pytest.mark.parametrize("mode,best", [(m, 0) for m in range(_hiplib.MODE_COUNT)] +
                         [(_hiplib.MODE_EXP_DIRECT, 256), (_hiplib.MODE_EXP_FAST, 16)])
def test_the_librarys_own_choice_and_its_range_are_timed(monkeypatch, tmp_path, mode, best):
    monkeypatch.setenv("PYFSTAT_AMD_TUNE_CACHE", str(tmp_path / "tune.json"))
    monkeypatch.setattr(autotune, "_time_step",
                        lambda b, reps: 1.0 if b.rows[mode] == best else 2.0)
    b = FakeBatch({"rect_fast": 8})
    res = autotune.tune(b, candidates={mode: autotune.CANDIDATES[mode]}, device_name="dev")
    assert res[mode]["rows"] == best and b.rows[mode] == best


@pytest.mark.parametrize("mode,one,two", [
    (_hiplib.MODE_RECT_GENERIC, "rect_step", "rect_generic"),
    (_hiplib.MODE_EXP_DIRECT, "exp_walk", "exp_direct"),
])
def test_a_value_of_one_kernel_is_not_taken_for_another(mode, one, two):
    keys = [autotune.shape_class(FakeBatch(k), mode, "dev")
            for k in ({one: 8}, {two: 8}, {one: 4, two: 4})]
    assert len(set(keys)) == 3
    # nor one of short steps for long ones
    keys.append(autotune.shape_class(FakeBatch({one: 8}, dtau=20 * 1800), mode, "dev"))
    assert keys[3] not in keys[:3]
    # the other modes' kernels do not matter
    assert keys[0] == autotune.shape_class(FakeBatch({one: 8, "rect_fast": 3}), mode, "dev")
