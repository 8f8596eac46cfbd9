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
