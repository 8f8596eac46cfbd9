"""B (sk_bp), A^T (sk_bp_adjoint) and B^T (sk_bp_transpose) on the fast kernels: every tile height,
bins off unit width (one to five candidates per pixel), axes off the detector's middle, degenerate
lines and sizes that no tile divides, against the oracle's matrices in FP64.

Tolerance: every entry is an FP32 length within about 4 ulp of the oracle's, and the sums of at
most 2 A (A^T) or 2 N (B^T) such products round to within a few 1e-7 of the FP64 sum in the
2-norm; 2e-6 leaves a factor of a few."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu

AXIS = np.array([0.0, 1.5707964, 0.7853982, 2.3561945, 1e-4, 1.5704], np.float32)
CASES = [
    ("two_pixels", 2, np.array([0.0, 0.3, 1.6], np.float32), 5, -2.0, 1.0),
    ("axis", 30, AXIS, 45, -22.0, 1.0),
    ("ragged", 70, (np.arange(67) * np.pi / 67).astype(np.float32), 101, -49.3, 1.0),
    ("half", 34, (np.arange(33) * np.pi / 33 + 0.01).astype(np.float32), 99, -24.0, 0.5),
    ("four_candidates", 50, (np.arange(41) * np.pi / 41).astype(np.float32), 180, -36.0, 0.4),
    ("five_candidates", 34, (np.arange(21) * np.pi / 21).astype(np.float32), 170, -25.2, 0.3),
    ("two_narrow", 66, (np.arange(53) * np.pi / 53).astype(np.float32), 103, -46.1, 0.9),
    ("wide", 66, (np.arange(40) * np.pi / 40).astype(np.float32), 48, -47.0, 2.0),
    # bin indices of 1.2e6 at half a bin: beyond the fast index (the kernels of exact mode run)
    ("far_axis", 32, (np.arange(3) * np.pi / 3 + 0.2).astype(np.float32), 1200100, -600000.0, 0.5),
]


@pytest.mark.parametrize("name,N,ang,R,rz,dr", CASES, ids=[c[0] for c in CASES])
@pytest.mark.parametrize("variant", [0, 1, 2])
def test_operators_against_the_oracles_matrices(ctx, name, N, ang, R, rz, dr, variant):
    A = ang.size
    geo = ctx.geometry(ang, rz, dr, R, N)
    rng = np.random.default_rng(17)
    y = rng.standard_normal((2, A, R)).astype(np.float32)
    v = rng.standard_normal((2, N, N)).astype(np.float32)
    geo.set_variants(7, variant)
    try:
        aty = geo.bp_adjoint(torch.from_numpy(y).cuda()).cpu().numpy()
        btv = geo.bp_transpose(torch.from_numpy(v).cuda()).cpu().numpy()
        by = geo.bp(torch.from_numpy(y).cuda()).cpu().numpy()
    finally:
        geo.set_variants(-1, -1)
    rp, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    B = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(N * N, A * R))
    for k in range(2):
        ref = oracle.fp_adjoint(ang, rz, dr, R, N, y[k].ravel())
        if np.any(ref):
            assert rel_l2(aty[k].ravel(), ref) <= 2e-6
        else:
            assert not np.any(aty[k])
        ref = B @ y[k].ravel().astype(np.float64)
        if np.any(ref):
            assert rel_l2(by[k].ravel(), ref) <= 2e-6
        else:
            assert not np.any(by[k])
        ref = B.T @ v[k].ravel().astype(np.float64)
        if np.any(ref):
            assert rel_l2(btv[k].ravel(), ref) <= 2e-6
        else:
            assert not np.any(btv[k])


# Rays that cut less than two pixels' length off a corner: a SIRT step's gradient divides them by
# that length, so each has to be right by itself.  An image of ones: at most 8 entries, each within
# about 4 ulp of the oracle's (4.8e-7), and 8 additions: 1e-6; 2e-6 leaves a factor of two.
@pytest.mark.parametrize("N,A,R,rz,dr", [(250, 142, 284, -174.9, 1.25), (64, 200, 91, -45.37, 1.0),
                                         (130, 97, 740, -92.2, 0.25), (2, 31, 21, -2.0, 0.2)])
def test_transpose_of_short_rays(ctx, N, A, R, rz, dr):
    ang = (np.arange(A) * np.pi / A + 0.1).astype(np.float32)
    geo = ctx.geometry(ang, rz, dr, R, N)
    got = geo.bp_transpose(torch.ones(N, N, device="cuda")).cpu().numpy().ravel()
    rp, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    ref = np.bincount(c, weights=vals.astype(np.float64), minlength=A * R)
    short = (ref > 0) & (ref < 2)
    assert short.sum() > 10
    np.testing.assert_allclose(got[short], ref[short], rtol=2e-6)
