"""sirt_batched with several images per work item: the item sizes that its rule picks, slices that leave a
remainder, and bin widths mixed, bit for bit against each slice alone."""
import math
import re

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _group(ctx, N, A, drho, batch, gen):
    R = math.ceil(math.sqrt(2) * N / drho)
    geo = ctx.geometry((np.arange(A) * math.pi / A).astype(np.float32), -(R - 1) / 2 * drho + 0.3, drho, R, N)
    return geo, torch.zeros(batch, N, N, device="cuda"), torch.rand(batch, A, R, device="cuda", generator=gen)


def _items(capfd):
    """Images per forward and per backprojector item, from the library's verbose line."""
    m = re.findall(r"fp mode \d+ x (\d+) images .* tiles x (\d+) images", capfd.readouterr().err)
    return tuple(int(v) for v in m[-1])


# groups of (N, angles, bin width, images) and the images per backprojector item that the rule has to
# pick for them: unit widths, one candidate a pixel beside two, three and four beside others
SETS = [
    ([(440, 37, 1.0, 11), (96, 20, 1.0, 3)], 4),
    ([(440, 37, 1.0, 15), (96, 20, 1.0, 5)], 8),
    ([(440, 37, 2.0, 15), (128, 20, 1.0, 9)], 8),
    ([(440, 37, 0.5, 11), (96, 20, 1.0, 6)], 4),
    ([(440, 37, 0.36, 15), (200, 20, 2.0, 5), (130, 20, 0.5, 7)], 4),
]


@pytest.mark.parametrize("sizes,images", SETS)
def test_items_of_several_images(ctx, monkeypatch, capfd, sizes, images):
    from synkrotomo_amd.projector import sirt_batched
    monkeypatch.setenv("SYNKRO_VERBOSE", "1")
    gen = torch.Generator(device="cuda").manual_seed(len(sizes))
    groups = [_group(ctx, *s, gen) for s in sizes]
    sirt_batched(groups, 2)
    assert _items(capfd)[1] == images
    for geo, x, sino in groups:
        for i in {0, images - 1, x.shape[0] - 1} & set(range(x.shape[0])):
            one = torch.zeros(geo.N, geo.N, device="cuda")
            geo.sirt_(one, sino[i].contiguous(), 2)
            assert torch.equal(x[i], one), (geo.N, i)


# A measurement that is not finite reaches the pixels its ray is a candidate of, and no others: a group
# whose pixels have fewer candidates than another group's takes only its own.
@pytest.mark.parametrize("batch", [1, 12])
def test_values_that_are_not_finite_stay_with_their_candidates(ctx, batch):
    from synkrotomo_amd.projector import sirt_batched
    gen = torch.Generator(device="cuda").manual_seed(2)
    groups = [_group(ctx, *s, batch, gen) for s in ((256, 29, 0.4), (230, 31, 2.0), (200, 23, 0.5), (96, 17, 1.0))]
    for geo, x, sino in groups:
        sino[0, 3, geo.R // 2] = math.inf
        sino[-1, 5, geo.R // 3] = math.nan
    sirt_batched(groups, 1)
    for geo, x, sino in groups:
        for i in {0, batch - 1}:
            one = torch.zeros(geo.N, geo.N, device="cuda")
            geo.sirt_(one, sino[i].contiguous(), 1)
            same = (x[i] == one) | (x[i].isnan() & one.isnan())
            assert bool(same.all()), (geo.N, i, int((~same).sum()))
            assert 0 < int((~x[i].isfinite()).sum()) < geo.N * geo.N // 4
