"""B^T (sk_bp_transpose) where the rays it walks by itself meet those it takes from A.x, against the
oracle's matrix in FP64."""
import numpy as np
import pytest
import scipy.sparse as sp
import torch

import oracle
from conftest import rel_l2

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


# Pixels that are not finite, and neighbours of either sign whose difference overflows: a ray is as the
# matrix has it -- infinite or NaN where it crosses such a pixel, and elsewhere the sum of the
# pixels it does cross -- in every kernel of A.x (the image in LDS, one image, four at a time, per
# wave).  No angle is a multiple of 45 degrees, so no ray lies on pixel edges or corners.  Finite
# rays: 4.8e-7 and 6e-8 per addition of the sum of magnitudes, at most 3 N / 2 entries.
@pytest.mark.parametrize("N,A,R,dr,batch,variant", [(64, 20, 91, 1.0, 1, -1), (130, 30, 185, 1.0, 1, 7),
                                                    (130, 30, 140, 1.4, 1, 3), (440, 37, 631, 1.0, 5, -1),
                                                    (66, 11, 420, 0.25, 2, -1)])
def test_transpose_of_pixels_that_are_not_finite(ctx, N, A, R, dr, batch, variant):
    ang = ((np.arange(A) + 0.37) * np.pi / A).astype(np.float32)
    rz = -(R - 1) / 2 * dr + 0.3
    rng = np.random.default_rng(N)
    v = rng.standard_normal((batch, N, N)).astype(np.float32)
    v[0, N // 2, N // 3] = np.inf
    v[0, N // 4, N // 2 + 1] = -np.inf
    v[0, 0, 0] = np.inf
    v[-1, N // 3, N // 2] = np.nan
    v[-1, N - 2, 1:3] = 2e38, -2e38
    geo = ctx.geometry(ang, rz, dr, R, N)
    geo.set_variants(variant, -1)
    try:
        got = geo.bp_transpose(torch.from_numpy(v).cuda()).cpu().numpy().reshape(batch, -1)
    finally:
        geo.set_variants(-1, -1)
    rp, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    rows = np.repeat(np.arange(N * N), np.diff(rp))
    keep = vals > 0
    for k in range(batch):
        x = v[k].ravel().astype(np.float64)[rows[keep]]
        w = vals[keep].astype(np.float64)
        bad = np.bincount(c[keep], weights=~np.isfinite(x), minlength=A * R) > 0
        np.testing.assert_array_equal(~np.isfinite(got[k]), bad)
        x = np.where(np.isfinite(x), x, 0)
        ref = np.bincount(c[keep], weights=w * x, minlength=A * R)
        mag = np.bincount(c[keep], weights=w * np.abs(x), minlength=A * R)
        assert np.all(np.abs(got[k] - ref)[~bad] <= (4.8e-7 + 1.5 * N * 6e-8) * mag[~bad])


# Pixels at whose outermost ray the candidate index rounds: on lines that are not degenerate A^T and B
# have the same lengths, and both follow the reference's index, so A^T r is the oracle's B r and B^T v
# its B^T v, at the largest |rhozero| as well as where the fast paths end (4 N) and just past them.
# Tolerance as in test_gpu_adjoints.py.
@pytest.mark.parametrize("N,rz,dr", [(64, -999000.3, 1.0), (64, -943000.7, 0.9), (32, -524000.2, 0.5), (64, -999900.3, 2.0),
                                     (64, -255.9, 1.0), (64, -256.1, 1.0), (64, -255.9, 0.25)])
def test_transpose_and_adjoint_with_the_references_candidates(ctx, N, rz, dr):
    ang = (np.pi / 4 + np.array([-0.05, -0.011, -0.003, 0.0007, 0.004, 0.02])).astype(np.float32)
    A, R = ang.size, int((-rz + N) / dr)
    rng = np.random.default_rng(3)
    y = rng.standard_normal((A, R)).astype(np.float32)
    v = rng.standard_normal((N, N)).astype(np.float32)
    geo = ctx.geometry(ang, rz, dr, R, N)
    aty = geo.bp_adjoint(torch.from_numpy(y).cuda()).cpu().numpy().ravel()
    btv = geo.bp_transpose(torch.from_numpy(v).cuda()).cpu().numpy().ravel()
    rp, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    B = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(N * N, A * R))
    assert rel_l2(aty, B @ y.ravel().astype(np.float64)) <= 2e-6
    assert rel_l2(btv, B.T @ v.ravel().astype(np.float64)) <= 2e-6


# Small images walk every line with the backprojector's lengths until a batch fills the chip; both ways
# on each side of the line, with degenerate lines and without.  Tolerance as in test_gpu_adjoints.py.
@pytest.mark.parametrize("N,A,first,batch", [(22, 16, 0.013, 1), (24, 16, 0.013, 1), (30, 21, 0.0, 1), (32, 21, 0.0, 1),
                                             (16, 22, 0.0, 128), (16, 22, 0.0, 129)])
def test_transpose_of_small_images(ctx, N, A, first, batch):
    ang = (np.arange(A) * np.pi / A + first).astype(np.float32)
    R = int(np.ceil(np.sqrt(2.0) * N)) + 1
    rz = -(R - 1) / 2 + 0.2
    v = np.random.default_rng(N).standard_normal((batch, N, N)).astype(np.float32)
    geo = ctx.geometry(ang, rz, 1.0, R, N)
    got = geo.bp_transpose(torch.from_numpy(v).cuda()).cpu().numpy()
    rp, c, vals = oracle.bp_csr(ang, rz, 1.0, R, N)
    B = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(N * N, A * R))
    for k in {0, batch // 2, batch - 1}:
        assert rel_l2(got[k].ravel(), B.T @ v[k].ravel().astype(np.float64)) <= 2e-6


# Diagonal rays an ulp off the pixels' corners: x_bot just below a pixel, x_top rounded up to its far edge,
# so the two ends' pixels are not the one the ray crosses.  By the walk of every ray (small images,
# exact mode), by A.x and its single rays.  Tolerance as in test_gpu_adjoints.py, in exact mode too
# (the sums' order is not the oracle's).
@pytest.mark.parametrize("exact_mode", [False, True], ids=["fast", "exact"])
@pytest.mark.parametrize("N,dr,rz,R", [(20, 0.70710677, -14.849242, 43), (22, 0.35355338, -16.617008, 94),
                                       (22, 1.4142135, -16.970562, 24), (30, 0.70710677, -22.627417, 64),
                                       (64, 0.35355338, -48.08326, 272), (64, 0.3, -11.7, 64)])
def test_transpose_on_diagonal_rays(ctx, N, dr, rz, R, exact_mode):
    ang = np.array([np.pi / 4, 3 * np.pi / 4, 5 * np.pi / 4, -np.pi / 4], np.float32)
    v = np.random.default_rng(1).standard_normal((N, N)).astype(np.float32)
    geo = ctx.geometry(ang, rz, dr, R, N)
    ctx.exact = exact_mode
    try:
        got = geo.bp_transpose(torch.from_numpy(v).cuda()).cpu().numpy().ravel()
        ones = geo.bp_transpose(torch.ones(N, N, device="cuda")).cpu().numpy().ravel()
    finally:
        ctx.exact = False
    rp, c, vals = oracle.bp_csr(ang, rz, dr, R, N)
    B = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(N * N, ang.size * R))
    assert rel_l2(got, B.T @ v.ravel().astype(np.float64)) <= 2e-6
    assert rel_l2(ones, B.T @ np.ones(N * N)) <= 2e-6


# The same rays in A^T: A gives such a row's whole length to the pixel of x_bot, B to the one between, and
# lines of each kind stand next to them in the table (other slopes, degenerate ones).  One image in
# the three tile heights, and 2, 4 and 8 at once (66^2 and 80^2 of two candidates).  Tolerance as in
# test_gpu_adjoints.py.
@pytest.mark.parametrize("variant,batch", [(0, 1), (1, 1), (2, 1), (-1, 52), (-1, 80), (-1, 280)])
@pytest.mark.parametrize("N,dr,rz,R", [(20, 1.4142135, -14.142135, 21), (80, 2.828427, -55.154327, 41),
                                       (80, 0.70710677, -21.92031, 64), (80, 0.35355338, -10.960155, 64),
                                       (66, 1.0, -30.292893, 63), (40, 0.4, -12.4, 64), (80, 1.25, -39.292893, 65)])
def test_adjoint_on_diagonal_rays(ctx, N, dr, rz, R, variant, batch):
    diag = [np.pi / 4, 3 * np.pi / 4, 5 * np.pi / 4, -np.pi / 4]
    ang = np.array(sorted(diag + [d + e for d in diag for e in (-0.3, -0.005, -0.0005, 0.0005, 0.005, 0.3)] + [0.0, np.pi / 2]),
                   np.float32)
    A = ang.size
    y = np.random.default_rng(2).standard_normal((batch, A, R)).astype(np.float32)
    geo = ctx.geometry(ang, rz, dr, R, N)
    geo.set_variants(-1, variant)
    try:
        got = geo.bp_adjoint(torch.from_numpy(y).cuda()).cpu().numpy().reshape(batch, -1)
    finally:
        geo.set_variants(-1, -1)
    rp, c, vals = oracle.fp_csr(ang, rz, dr, R, N)
    At = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(A * R, N * N)).T
    for k in {0, batch // 2, batch - 1}:
        assert rel_l2(got[k], At @ y[k].ravel().astype(np.float64)) <= 2e-6


# Few lines of few pixels run A^T's general kernel: both sides of each line of that rule (12 lines up to
# 2^18 pixels, 8 up to 2^20, 5 of narrow bins).  Tolerance as in test_gpu_adjoints.py.
@pytest.mark.parametrize("N,batch,A,dr", [(2, 1, 1, 1.0), (64, 64, 12, 1.0), (64, 65, 12, 1.0), (64, 64, 13, 2.0), (64, 65, 8, 2.0),
                                          (64, 255, 8, 1.0), (64, 256, 8, 1.0), (66, 30, 5, 0.4), (66, 30, 6, 0.4), (64, 256, 5, 0.4)])
def test_adjoint_of_few_lines(ctx, N, batch, A, dr):
    ang = ((np.arange(A) + 0.2) * np.pi / A).astype(np.float32)
    R = int(np.ceil(np.sqrt(2.0) * N / dr))
    rz = -(R - 1) / 2 * dr + 0.1
    y = np.random.default_rng(A).standard_normal((batch, A, R)).astype(np.float32)
    got = ctx.geometry(ang, rz, dr, R, N).bp_adjoint(torch.from_numpy(y).cuda()).cpu().numpy().reshape(batch, -1)
    rp, c, vals = oracle.fp_csr(ang, rz, dr, R, N)
    At = sp.csr_matrix((vals.astype(np.float64), c, rp), shape=(A * R, N * N)).T
    for k in {0, batch // 2, batch - 1}:
        assert rel_l2(got[k], At @ y[k].ravel().astype(np.float64)) <= 2e-6
