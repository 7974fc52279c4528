"""The merge and prefix kernel at the edges of its workgroup shapes: bins per
round, several rounds, bins without and with many atoms, detectors."""

import numpy as np
import pytest

from pyfstat_amd import synth
from pyfstat_amd.atoms import TRANSIENT_RECTANGULAR, transientWindowRange_t

pytestmark = pytest.mark.gpu

TA = synth.TSFT


def _template(rng, N, n_det, kind):
    """Atoms of one template on N bins: (ts, cols) per detector."""
    out = []
    for X in range(n_det):
        if kind == "dense":  # up to 5 atoms a bin
            bins = np.sort(rng.integers(0, N, 3 * N))
        elif kind == "gap":  # most bins empty, whole rounds too
            bins = np.sort(rng.integers(0, N, max(2, N // 50)))
        else:
            bins = np.arange(N)
        bins[0], bins[-1] = 0, N - 1
        ts = np.sort(bins * TA + rng.integers(0, TA // 4, bins.size))
        ts[0] = 0
        cols = rng.normal(0, 1, (7, ts.size)).astype(np.float32)
        cols[:2] = rng.uniform(0.5, 1.5, (2, ts.size))
        cols[2] = 0.3 * rng.uniform(-1, 1, ts.size) * np.sqrt(cols[0] * cols[1])  # cond < 10
        out.append(((synth.T_START + ts).astype(np.uint32), cols))
    return out


def _prefix(tmpl, N, t_min):
    """Merged float32 bins (detectors and atoms in order) and their FP64 prefix."""
    bins = np.zeros((N, 7), np.float32)
    for ts, cols in tmpl:
        b = (ts.astype(np.int64) - t_min) // TA
        for k in np.flatnonzero(b < N):
            bins[b[k]] += cols[:, k]
    return np.vstack([np.zeros((1, 7)), np.cumsum(bins.astype(np.float64), axis=0)])


@pytest.mark.parametrize("few", [True, False])
@pytest.mark.parametrize("kind,n_det", [("full", 1), ("full", 2), ("dense", 3), ("gap", 10)])
def test_prefix_at_workgroup_edges(hip_ready, few, kind, n_det):
    from pyfstat_amd.batched import BatchedTransientMaps

    rng = np.random.default_rng(len(kind) * 16 + n_det)
    sizes = [2, 3, 127, 509, 511, 512, 513, 1023, 1024, 1025, 2049, 4096, 4097, 5000]
    # more long templates than the wide workgroups take
    sizes += [] if few else [1030] * 660
    tmpls = [_template(rng, N, n_det, kind) for N in sizes[:14]]
    tmpls += [tmpls[9]] * (len(sizes) - 14)
    flat = [d for t in tmpls for d in t]
    off = np.concatenate([[0], np.cumsum([ts.size for ts, _ in flat])])
    wins, ref = [], {}
    for t, tmpl in enumerate(tmpls):
        t_min = min(int(ts[0]) for ts, _ in tmpl)
        N = (max(int(ts[-1]) for ts, _ in tmpl) - t_min) // TA + 1
        n = min(N - 1, 40)
        # starts over all the data, two windows each of at least two bins
        dt0 = max(1, (N - 2) // n) * TA
        wins.append(transientWindowRange_t(type=TRANSIENT_RECTANGULAR, t0=t_min,
                                           t0Band=(n - 1) * dt0, dt0=dt0, tau=2 * TA,
                                           tauBand=max(N // 2, 1) * TA, dtau=max(N // 2, 1) * TA))
        if t < 14:
            ref[t] = (_prefix(tmpl, N, t_min), N, n, dt0 // TA)
    b = BatchedTransientMaps(np.concatenate([ts for ts, _ in flat]),
                             np.concatenate([c for _, c in flat], axis=1), off,
                             np.arange(len(tmpls) + 1, dtype=np.int64) * n_det, wins, TA,
                             BtSG=True)
    b.run()
    F = b.F_host()
    lo = 0
    for t in range(14):
        P, N, n, step = ref[t]
        want = np.zeros((n, 2))
        for m in range(n):
            for j in range(2):
                i0, i1 = m * step, min(m * step + 2 + j * max(N // 2, 1) - 1, N - 1)
                A, B, C, ar, ai, br, bi = P[i1 + 1] - P[i0]
                D = A * B - C * C
                want[m, j] = (B * (ar**2 + ai**2) + A * (br**2 + bi**2)
                              - 2 * C * (ar * br + ai * bi)) / D if D > 0 else 2.0
        got = F[lo:lo + 2 * n].reshape(n, 2).astype(np.float64)
        lo += 2 * n
        # well-conditioned cells: a handful of float32 roundings (6e-8 each), and
        # window sums 20 x 2^-53 of prefixes below 2e4 off
        np.testing.assert_allclose(got, want, rtol=2e-6, atol=1e-9, err_msg=str((t, N)))
    for t in range(15, len(tmpls)):  # equal templates, equal maps, in any workgroup
        k = lo + (t - 14) * 80
        np.testing.assert_array_equal(F[k:k + 80], F[lo:lo + 80])
    b.close()
