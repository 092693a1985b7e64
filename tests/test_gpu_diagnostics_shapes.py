"""Device ESS and R-hat at the edges of the blocked lag sums.

The blocked kernel takes 64 coordinates (or chains) a wave, 32 lags a
workgroup and series of up to 289 samples; these shapes sit on, below and above
those limits, in the axis orders and types that callers use.  Against the
oracle's FFT estimators: 1e-10 (ESS) and 1e-12 (R-hat) relative, as the other
diagnostics tests (float64 sums of at most 1e6 terms of order one).
"""
import numpy as np
import pytest
import torch

import geomjax_amd as gj
from oracle import diagnostics as od
from tests.helpers import rel_err, seeded_normal

pytestmark = pytest.mark.gpu


def _series(T, C, D, seed):
    z = seeded_normal(seed, T, C, D)
    x = z.clone()
    for t in range(1, T):
        x[t] = 0.7 * x[t - 1] + z[t]
    return x


@pytest.mark.parametrize("T,C,D", [
    (2, 2, 64), (7, 40, 1), (8, 33, 3), (31, 3, 65), (32, 70, 31), (33, 64, 32), (100, 1030, 64), (100, 129, 2),
    (289, 40, 33), (290, 40, 33), (257, 2100, 5)])
@pytest.mark.parametrize("dtype", [torch.float64, torch.float32])
def test_ess_and_rhat_match_oracle(T, C, D, dtype):
    print(f"case T={T} C={C} D={D} {dtype}", flush=True)
    x = _series(T, C, D, T + C + D).to(dtype)
    ref = x.double().numpy()
    e, r = od.effective_sample_size(ref, 1, 0), od.potential_scale_reduction(ref, 1, 0)
    d = x.to("cuda:0")
    assert rel_err(gj.ess(d, chain_axis=1, sample_axis=0), np.atleast_1d(e).reshape(e.shape)) < 1e-10
    assert rel_err(gj.rhat(d, chain_axis=1, sample_axis=0), r) < 1e-12
    # the sample axis innermost, and a strided view
    p = d.permute(1, 2, 0).contiguous()
    assert rel_err(gj.ess(p, chain_axis=0, sample_axis=2), e) < 1e-10
    wide = torch.zeros(T, C, 2 * D, dtype=dtype, device="cuda:0")
    wide[:, :, ::2] = d
    assert rel_err(gj.ess(wide[:, :, ::2], chain_axis=1, sample_axis=0), e) < 1e-10
