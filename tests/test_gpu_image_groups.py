"""Kernels that work on several images at once (A.x 4 or 2 images per workgroup, B.r, A^T.r and the
SIRT update 8, 4 or 2) give each image the bits it gets alone: batches around the group sizes,
every staged width of A.x (chunks of 64 columns: bin widths 1, 1.3 and 2), groups of fewer than
four lines, a ragged last bin block and tile row, tiles with and without the exact step.
The images hold both signs and, in one case, values far apart."""
import math

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu

# name, N, angles, bins, first angle, bin width; enough workgroups that batches run grouped
GEOMETRIES = [
    ("two_chunks", 64, 701, 93, 0.0, 1.0),
    ("three_chunks", 96, 803, 130, 0.01, 1.3),
    ("four_chunks", 128, 901, 130, 0.4, 2.0),
]


def _geometry(ctx, N, A, R, start, drho):
    ang = (start + np.arange(A) * math.pi / A).astype(np.float32)
    return ctx.geometry(ang, -(R - 1) / 2 * drho + 0.3, drho, R, N)


@pytest.mark.parametrize("name,N,A,R,start,drho", GEOMETRIES, ids=[g[0] for g in GEOMETRIES])
@pytest.mark.parametrize("batch", [2, 3, 5, 8])
def test_projection_of_a_batch_is_each_images_own(ctx, name, N, A, R, start, drho, batch):
    geo = _geometry(ctx, N, A, R, start, drho)
    gen = torch.Generator(device="cuda").manual_seed(batch)
    x = torch.randn(batch, N, N, device="cuda", generator=gen)
    x[-1] *= 1e6
    geo.set_variants(7, 2)
    try:
        got = geo.fp(x)
        geo.set_variants(0, 2)  # one ray per lane, one image per launch block
        for k in range(batch):
            assert torch.equal(got[k], geo.fp(x[k].contiguous())), k
    finally:
        geo.set_variants(-1, -1)


# images held in LDS (up to 80^2, few workgroups) against the per-wave kernel: sizes around a wave
# and a workgroup, the largest and the first past it, bins past both edges of the image,
# fewer items than waves, batches on both sides of the bound on workgroups
@pytest.mark.parametrize("N,A,R,drho,batch", [(2, 1, 3, 1.0, 1), (6, 5, 9, 0.5, 2), (62, 7, 200, 0.7, 1),
                                              (64, 90, 91, 1.0, 1), (64, 90, 91, 1.0, 17), (64, 90, 91, 1.0, 18),
                                              (78, 33, 64, 2.5, 3), (80, 126, 65, 1.0, 2), (82, 20, 117, 1.0, 2)])
def test_small_images_in_lds_give_the_per_wave_kernels_bits(ctx, N, A, R, drho, batch):
    geo = _geometry(ctx, N, A, R, 0.0, drho)
    gen = torch.Generator(device="cuda").manual_seed(N)
    x = torch.randn(batch, N, N, device="cuda", generator=gen)
    x[-1] *= 1e6
    b = torch.rand(batch, A, R, device="cuda", generator=gen)
    got, step = geo.fp(x), geo.sirt_(x.clone(), b, 2)
    geo.set_variants(3, 0)
    try:
        assert torch.equal(got, geo.fp(x))
        assert torch.equal(step, geo.sirt_(x.clone(), b, 2))
    finally:
        geo.set_variants(-1, -1)


# the batches run 2, 4, 4, 4, 4 and 8 images per workgroup at 440^2 (28 x 14 tiles of 16 x 32); bins
# of 0.9 have two candidates per pixel too, of 0.4, 0.5 and 2 four, three and one (4 images or 1)
@pytest.mark.parametrize("batch,drho", [(2, 1.0), (3, 1.0), (6, 1.0), (11, 1.0), (16, 0.9), (40, 1.0), (2, 0.5), (6, 0.4),
                                        (6, 0.5), (6, 2.0)])
@pytest.mark.parametrize("op", ["bp", "bp_adjoint"])
def test_backprojection_of_a_batch_is_each_images_own(ctx, op, batch, drho):
    N, A, R = 440, 37, math.ceil(631 / drho)
    geo = _geometry(ctx, N, A, R, 0.0, drho)
    gen = torch.Generator(device="cuda").manual_seed(batch)
    y = torch.randn(batch, A, R, device="cuda", generator=gen)
    y[-1] *= 1e6
    got = getattr(geo, op)(y)
    geo.set_variants(7, 2)
    try:
        for k in range(batch):
            assert torch.equal(got[k], getattr(geo, op)(y[k].contiguous())), k
    finally:
        geo.set_variants(-1, -1)


@pytest.mark.parametrize("batch", [9, 40])  # 4 and 8 images per workgroup
def test_sirt_update_of_a_batch_is_each_slices_own(ctx, batch):
    N, A, R = 440, 37, 631
    geo = _geometry(ctx, N, A, R, 0.0, 1.0)
    b = torch.rand(batch, A, R, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    x = torch.zeros(batch, N, N, device="cuda")
    geo.sirt_(x, b, 3)
    for k in range(batch):
        one = torch.zeros(N, N, device="cuda")
        geo.sirt_(one, b[k].contiguous(), 3)
        assert torch.equal(x[k], one), k


@pytest.mark.parametrize("batch", [2, 3, 6])
def test_sirt_of_a_batch_is_each_slices_own(ctx, batch):
    name, N, A, R, start, drho = GEOMETRIES[0]
    geo = _geometry(ctx, N, A, R, start, drho)
    gen = torch.Generator(device="cuda").manual_seed(7)
    b = torch.rand(batch, A, R, device="cuda", generator=gen)
    x = torch.zeros(batch, N, N, device="cuda")
    geo.set_variants(7, 2)
    try:
        geo.sirt_(x, b, 3)
        geo.set_variants(0, 0)
        for k in range(batch):
            one = torch.zeros(N, N, device="cuda")
            geo.sirt_(one, b[k].contiguous(), 3)
            assert torch.equal(x[k], one), k
    finally:
        geo.set_variants(-1, -1)


# (groups of (N, angles, bins, bin width), images per group): items of 1, 2, 4 and 8 images, groups
# that leave a remainder, bin widths with one to four candidates mixed, and the narrow bins of the
# general path
BATCHES = [
    ([(128, 200, 182, 1.0), (96, 150, 137, 1.0)], 2),
    ([(128, 200, 182, 1.0), (96, 150, 137, 1.0), (200, 90, 283, 1.0)], 7),
    ([(256, 400, 363, 1.0), (64, 90, 91, 1.0)], 9),
    ([(256, 400, 363, 1.0), (128, 120, 400, 0.5), (130, 77, 100, 2.0), (96, 60, 350, 0.4)], 5),
    ([(64, 90, 320, 0.3)], 3),
]


@pytest.mark.parametrize("sizes,batch", BATCHES)
def test_batched_sirt_equals_each_slice_alone(ctx, sizes, batch):
    from synkrotomo_amd.projector import sirt_batched
    gen = torch.Generator(device="cuda").manual_seed(batch)
    groups = []
    for k, (N, A, R, drho) in enumerate(sizes):
        geo = _geometry(ctx, N, A, R, 0.0, drho)
        b = batch + (k == 1)
        groups.append((geo, torch.zeros(b, N, N, device="cuda"), torch.rand(b, A, R, device="cuda", generator=gen)))
    sirt_batched(groups, 3)
    for geo, x, sino in groups:
        for i in (0, x.shape[0] - 1):
            one = torch.zeros(geo.N, geo.N, device="cuda")
            geo.sirt_(one, sino[i].contiguous(), 3)
            assert torch.equal(x[i], one), (geo.N, i)
