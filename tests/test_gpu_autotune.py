"""What the autotuner times."""
import math
import re

import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _geometry(ctx, N, A):
    R = math.ceil(math.sqrt(2) * N)
    return ctx.geometry((np.arange(A) * math.pi / A).astype(np.float32), -(R - 1) / 2, 1.0, R, N)


# The backprojector's variants are tile heights of one image: where a batch runs several images per
# workgroup they are all the same kernel, so they are timed on the largest batch that does not.
@pytest.mark.parametrize("N,A,batch,timed", [(256, 180, 32, 4), (256, 180, 2, 2), (512, 40, 8, 1), (64, 40, 16, 16)])
def test_backprojector_variants_are_timed_where_they_differ(ctx, monkeypatch, capfd, N, A, batch, timed):
    monkeypatch.setenv("SYNKRO_VERBOSE", "1")
    geo = _geometry(ctx, N, A)
    capfd.readouterr()
    try:
        geo.autotune(batch)
    finally:
        geo.set_variants(-1, -1)
    lines = re.findall(r"bp variant (\d), (\d+) images", capfd.readouterr().err)
    assert lines == [(str(v), str(timed)) for v in range(3)]


# Images up to 80^2 have a forward kernel that is no variant: it is timed beside them, and where it wins
# the geometry stays without a variant, so tuning never makes such a projection slower.
@pytest.mark.parametrize("N,batch,timed", [(64, 1, True), (80, 2, True), (64, 256, False), (96, 1, False)])
def test_small_images_kernel_is_timed_beside_the_variants(ctx, monkeypatch, capfd, N, batch, timed):
    monkeypatch.setenv("SYNKRO_VERBOSE", "1")
    geo = _geometry(ctx, N, 90)
    capfd.readouterr()
    try:
        best = geo.autotune(batch)[0]
    finally:
        geo.set_variants(-1, -1)
    lines = re.findall(r"fp variant (-?\d+): ([\d.]+) ms", capfd.readouterr().err)
    assert [int(v) for v, _ in lines] == list(range(-1 if timed else 0, 8))
    # the fastest is kept (times are printed to a microsecond)
    assert float(dict(lines)[str(best)]) == min(float(t) for _, t in lines)
