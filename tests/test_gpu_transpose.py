"""B^T (sk_bp_transpose) where the rays it walks by itself meet those it takes from A.x, against the
oracle's matrix in FP64."""
import numpy as np
import pytest
import torch

import oracle

pytestmark = pytest.mark.gpu


# An axis so far from the detector's first bin that FP32 bin numbers are off by more than the range of
# short chords of a nearly axis-parallel line: rays that cross many rows next to those that cross
# one.  An image of ones: at most 70 entries a ray, each within about 4 ulp of the oracle's (4.8e-7),
# and 70 additions (6e-8 each): 5e-6 of the sum; a ray that only cuts a corner may come from A.x,
# off by 6e-8 in each of its rows: 1e-5.
@pytest.mark.parametrize("N,rz,dr,R,angles", [
    (32, -138915.8125, 1.3, 106892, [3.143056631]),
    (64, -150000.03, 1.0, 150060, [0.0015, 1.5723, 3.1401]),
    (64, -300000.03, 1.0, 300060, [0.0015, 1.5723, 3.1401]),
    (64, -300000.03, 0.5, 600120, [0.0013, 1.5695]),
    (64, -255.97, 1.0, 300, [0.0011, 0.0015, 0.004, 1.5723, 1.5695, 3.1401]),
])
def test_transpose_far_from_the_detectors_first_bin(ctx, N, rz, dr, R, angles):
    ang = np.array(angles, np.float32)
    geo = ctx.geometry(ang, rz, dr, R, N)
    got = geo.bp_transpose(torch.ones(N, N, device="cuda")).cpu().numpy().ravel()
    _, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    ref = np.bincount(c, weights=vals.astype(np.float64), minlength=ang.size * R)
    assert (ref > 2).sum() > 20
    np.testing.assert_allclose(got, ref, rtol=5e-6, atol=1e-5)
