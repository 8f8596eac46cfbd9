"""The correction network's kernels at the ends of the sizes that they accept."""
import pytest
import torch

from synkrotomo_amd import _native as nat
from synkrotomo_amd.projector import _ptr, _stream

pytestmark = pytest.mark.gpu


# More images than workgroups of 256 threads fit a launch (2^24): single pixels, so that the gradient is
# the centre tap's product with the 32 channels.  Integers: every product and sum is exact.
def test_data_gradient_of_very_many_images(ctx):
    B = (1 << 24) + 77
    gen = torch.Generator(device="cuda").manual_seed(0)
    dh = torch.randint(-8, 9, (B, 32), device="cuda", generator=gen, dtype=torch.int8).to(torch.bfloat16)
    mask = torch.randint(-1, 2, (B, 32), device="cuda", generator=gen, dtype=torch.int8).to(torch.bfloat16)
    w = torch.randint(-4, 5, (32, 3, 3), device="cuda", generator=gen).to(torch.bfloat16)
    dx = torch.full((B,), torch.nan, device="cuda")
    nat.check(nat.lib().sk_conv_in_dgrad(ctx.handle, B, 1, 1, _ptr(dh), _ptr(mask), _ptr(w), _ptr(dx), _stream(0)),
              ctx.handle, "dgrad")
    for part in (slice(0, 4096), slice(1 << 20, (1 << 20) + 4096), slice(B - 4096, B)):
        ref = (dh[part].float() * (mask[part] > 0)) @ w[:, 1, 1].float()
        assert torch.equal(dx[part], ref)
    assert bool(dx.isfinite().all())
