"""A merge on a stream of its own, behind work queued there, whose result another
stream reads after waiting for it: values, bins and gradients."""

import numpy as np
import pytest

from tests.test_gpu_merge_plan import TA, _segments

pytestmark = pytest.mark.gpu


def test_merge_on_another_stream(hip_ready):
    import torch

    from pyfstat_amd.refine import MergedAtoms

    segs = _segments(9)
    dev = torch.device("cuda", 0)
    ts = np.concatenate([s for _, s in segs])
    off = np.concatenate([[0], np.cumsum([s.size for _, s in segs])])
    tmpl = np.array([t for t, _ in segs])
    begin = np.searchsorted(tmpl, np.arange(tmpl[-1] + 2))
    ts_d = torch.from_numpy(ts.view(np.int32)).to(dev)
    raw = torch.randn(7, ts.size, device=dev, generator=torch.Generator(dev).manual_seed(5))
    weight = torch.randn(7, 1, device=dev, generator=torch.Generator(dev).manual_seed(6))
    ref = MergedAtoms(ts_d, off, begin, TA, ts.size, dev)
    want = ref.merge(raw).clone()
    bins = ref.atom_bin.clone()
    torch.cuda.synchronize()
    side = torch.cuda.Stream()
    for _ in range(3):
        merged = MergedAtoms(ts_d, off, begin, TA, ts.size, dev)
        a = torch.randn(2048, 2048, device=dev)
        x = raw.clone().requires_grad_(True)
        side.wait_stream(torch.cuda.current_stream())
        with torch.cuda.stream(side):
            for _k in range(8):  # work that the merge waits behind
                a = a @ a * 1e-3
            got = merged.merge(x)
        torch.cuda.current_stream().wait_stream(side)
        (grad,) = torch.autograd.grad((got * weight).sum(), x)
        assert torch.equal(got, want) and torch.equal(merged.atom_bin, bins)
        assert torch.equal(grad, weight.expand(7, ts.size))
        del merged
