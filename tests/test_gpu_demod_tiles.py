"""Atoms of banks of templates at every tile width of the launch (8, 16, 32 and
64 templates a workgroup), with partial tiles of templates and of SFTs: sampled
templates against the FP64 oracle."""

import numpy as np
import pytest

from pyfstat_amd import synth
from tests.test_gpu_demod import _check_atoms

pytestmark = pytest.mark.gpu


# 5 tiles of SFTs: 64 templates a tile from 4000 tiles on, 32 from 3000 of its
# own, 16 from 1000
@pytest.mark.parametrize("T", [33, 1001, 4001, 20003, 51213])
@pytest.mark.parametrize("dterms", [8, 5])
def test_bank_of_templates(hip_ready, T, dterms):
    from pyfstat_amd.demod import demod_atoms

    sft = synth.synthetic_sfts(n_det=2, n_sft=130, gap_frac=0.0, seed_index=76)
    rng = np.random.default_rng(76 + T)
    freqs = rng.uniform(100.0, 100.05, T)
    fdots = rng.uniform(-5e-9, 5e-9, T)
    at = demod_atoms(sft.sft_set(), freqs, fdots, sft.ref_time, dterms=dterms)
    n = sft.t_start.size
    pick = np.unique([0, 1, 7, 8, 15, 16, 31, 32, T // 2, T - 2, T - 1])
    rows = (pick[:, None] * n + np.arange(n)).reshape(-1)
    import torch

    idx = torch.from_numpy(rows).to(at.cols_d.device)
    ts = at.ts_d[idx].cpu().numpy().view(np.uint32)
    cols = at.cols_d[:, idx].cpu().numpy()
    _check_atoms(ts, cols, sft, freqs[pick], fdots[pick], dterms)
