"""The batched merge as a plan of many runs: block and chunk edges, several
atoms a bin, gaps longer than a block, against a per-bin loop."""

import numpy as np
import pytest

from pyfstat_amd import synth

pytestmark = pytest.mark.gpu

TA = synth.TSFT


def _segments(seed):
    """(template, timestamps) of segments: one bin, 1023 to 1025 and 2600 bins,
    up to five atoms a bin (more atoms than a chunk holds), and a long gap."""
    rng = np.random.default_rng(seed)
    out = []
    for t, n in enumerate((1, 1023, 1024, 1025, 2600)):
        for _x in range(1 + t % 3):
            keep = np.sort(rng.choice(n, size=max(1, int(0.8 * n)), replace=False))
            if n > 2000:
                keep = keep[(keep < 40) | (keep > 1900)]
            reps = rng.integers(1, 6 if t == 3 else 2, size=keep.size)
            ts = np.repeat(keep, reps) * TA + rng.integers(0, TA, size=int(reps.sum()))
            ts = np.unique(np.append(ts, [0, (n - 1) * TA])) + synth.T_START
            out.append((t, ts.astype(np.uint32)))
    return out


def test_merge_runs_match_per_bin_sums(hip_ready):
    import torch

    from pyfstat_amd.refine import MergedAtoms

    segs = _segments(3)
    dev = torch.device("cuda", 0)
    ts = np.concatenate([s for _, s in segs])
    off = np.concatenate([[0], np.cumsum([s.size for _, s in segs])])
    tmpl = np.array([t for t, _ in segs])
    begin = np.searchsorted(tmpl, np.arange(tmpl[-1] + 2))
    rng = np.random.default_rng(4)
    merged = MergedAtoms(torch.from_numpy(ts.view(np.int32)).to(dev), off, begin, TA, ts.size, dev)
    side = torch.cuda.Stream()
    for k in range(3):  # the plan is run again, on other data and another stream
        cols = rng.standard_normal((7, ts.size)).astype(np.float32)
        with torch.cuda.stream(side if k == 1 else torch.cuda.current_stream()):
            got = merged.merge(torch.from_numpy(cols).to(dev)).cpu().numpy()
        ref = np.zeros((7, merged.total_bins), dtype=np.float32)
        want = np.empty(ts.size, dtype=np.int64)
        for s, (t, x) in enumerate(segs):
            b = merged.m_off[t] + (x.astype(np.int64) - int(merged.t_data[t])) // TA
            want[off[s]:off[s + 1]] = b
            for q, i in enumerate(b):  # float32, in atom order
                ref[:, i] += cols[:, off[s] + q]
        assert np.array_equal(got, ref)
        assert np.array_equal(merged.atom_bin.cpu().numpy(), want)
