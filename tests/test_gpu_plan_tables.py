"""Plans whose descriptors go to the device in one copy (small batches) and table by
table (large ones), with templates of every kernel between each other: the same
maps and statistics as each template's plan by itself."""

import numpy as np
import pytest

from tests.test_gpu_autotune_kernels import DISPATCH, _batch
from tests.test_gpu_rect_blocks import _atoms

pytestmark = pytest.mark.gpu

CASES = [c for c, _ in DISPATCH if not c[-1]]


# 192 bytes of descriptor a template: 256 KB lie between the two
@pytest.mark.parametrize("copies", [1, 100])
def test_mixed_batch_matches_single_templates(hip_ready, copies):
    ts, cols = _atoms(200, 3, "plain")
    b = _batch(CASES * copies, ts, cols)
    assert all(b.templates_per_kernel().values())
    b.run()
    F, st = b.F_host(), b.stats()
    for k, case in enumerate(CASES):
        one = _batch([case], ts, cols)
        one.run()
        G, (sg,) = one.F_host(), one.stats()
        one.close()
        for t in range(k, b.T, len(CASES)):
            m = b.map_view(F, t).reshape(-1)
            # the sums of the exponential windows depend on the items by 1e-13,
            # times the condition number (< 1e4), and F is a float32
            np.testing.assert_allclose(m, G, rtol=1e-6, atol=1e-7)
            assert st["maxF"][t] == m.max()
            assert st["m_ML"][t] * st["N_tau"][t] + st["n_ML"][t] == m.argmax()
            assert (st["N_t0"][t], st["N_tau"][t]) == (sg["N_t0"], sg["N_tau"])
            # 1e-6 of the sum, and F's rounding times F
            assert abs(st["lnBtSG"][t] - sg["lnBtSG"]) <= 2e-6 + 6e-7 * abs(sg["maxF"])
    b.close()
