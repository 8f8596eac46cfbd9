"""SIRT of stacks on the kernels that its sizes call for: off-width bins with several images per workgroup,
and iteration graphs that hold the kernels in force."""
import math
import re

import numpy as np
import pytest
import torch

pytestmark = pytest.mark.gpu


def _geometry(ctx, N, A, drho):
    R = math.ceil(math.sqrt(2) * N / drho)
    return ctx.geometry((np.arange(A) * math.pi / A).astype(np.float32), -(R - 1) / 2 * drho + 0.3, drho, R, N)


# 4 images per workgroup with 1, 2, 3 and 4 candidates a pixel, the last ones repeated
@pytest.mark.parametrize("drho", [2.0, 0.9, 0.5, 0.4])
def test_update_of_a_stack_is_each_slices_own(ctx, drho):
    geo = _geometry(ctx, 440, 37, drho)
    b = torch.rand(6, geo.A, geo.R, device="cuda", generator=torch.Generator(device="cuda").manual_seed(3))
    x = torch.zeros(6, 440, 440, device="cuda")
    geo.sirt_(x, b, 2)
    for k in (0, 3, 5):
        one = torch.zeros(440, 440, device="cuda")
        geo.sirt_(one, b[k].contiguous(), 2)
        assert torch.equal(x[k], one), k


# A geometry's variant 0 is a kernel, no variant is the rule by size: each has its own graph on the same
# buffers, and going back finds the first again.
def test_graphs_hold_the_variants_in_force(ctx, monkeypatch, capfd):
    monkeypatch.setenv("SYNKRO_VERBOSE", "1")
    geo = _geometry(ctx, 256, 40, 1.0)
    b = torch.rand(geo.A, geo.R, device="cuda")
    x = torch.zeros(256, 256, device="cuda")
    seen = []
    try:
        for variants in ((-1, -1), (0, 0), (-1, -1), (0, 0), (7, 2)):
            geo.set_variants(*variants)
            capfd.readouterr()
            geo.sirt_(x.zero_(), b, 8)
            seen.append(re.findall(r"fp variant (-?\d+), bp variant (-?\d+)", capfd.readouterr().err))
    finally:
        geo.set_variants(-1, -1)
    assert seen == [[("-1", "-1")], [("0", "0")], [], [], [("7", "2")]]
