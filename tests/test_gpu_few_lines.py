"""A.x of a geometry that was not tuned, on both sides of the lines that its choice of kernel draws for few
lines, against the oracle."""
import numpy as np
import pytest
import torch

import oracle
from conftest import rel_l2

pytestmark = pytest.mark.gpu


# One line; ten and eleven lines (N = 130: 3 waves a line); ten of fewer workgroups than 128; bins below 1,
# 8 pixels across a line and just more, several images per workgroup; a detector that is one bin.
# Tolerance: the projector's parity bound, as in test_gpu_projector.py.
@pytest.mark.parametrize("N,A,dr,batch", [(130, 1, 1.0, 1), (512, 1, 2.0, 2), (130, 10, 1.0, 16), (130, 10, 1.0, 15), (130, 11, 1.0, 16),
                                          (256, 32, 0.5, 16), (264, 32, 0.5, 16), (258, 32, 0.5, 16), (96, 12, 0.36, 64), (2, 3, 1.0, 512)])
def test_projection_of_few_lines(ctx, N, A, dr, batch):
    ang = (np.arange(A) * np.pi / A + 0.013).astype(np.float32)
    R = int(np.ceil(np.sqrt(2.0) * N / dr)) if N > 2 else 1
    rz = -(R - 1) / 2 * dr
    x = np.random.default_rng(A).standard_normal((batch, N, N)).astype(np.float32)
    got = ctx.geometry(ang, rz, dr, R, N).fp(torch.from_numpy(x).cuda()).cpu().numpy().reshape(batch, -1)
    for k in {0, batch // 2, batch - 1}:
        assert rel_l2(got[k], oracle.fp(ang, rz, dr, R, x[k])) <= 1e-5
