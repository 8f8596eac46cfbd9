"""Gradient kernels of the correction network on small integers, where every product and sum is
exact in FP32: weight and bias gradients of all four layer kinds and the data gradients of the first
layer, at one pixel, whole tiles, ragged tiles and more tiles than the launch has blocks."""
import pytest
import torch
import torch.nn.functional as F

pytestmark = pytest.mark.gpu

SIZES = [(1, 1, 1), (1, 16, 16), (2, 17, 33), (3, 48, 15), (5, 256, 256)]


def _ints(gen, shape, low, high, dtype):
    return torch.randint(low, high + 1, shape, device="cuda", generator=gen).to(dtype)


def _shifted(x, t):
    """x [B, H, W, C] at p + off_t, zero outside."""
    H, W = x.shape[1:3]
    return F.pad(x, (0, 0, 1, 1, 1, 1))[:, t // 3:t // 3 + H, t % 3:t % 3 + W]


@pytest.mark.parametrize("B,H,W", SIZES)
@pytest.mark.parametrize("kind,CO,CI", [(0, 32, 1), (1, 32, 32), (2, 1, 32), (3, 32, 2)])
def test_weight_gradients_are_exact_on_integers(ctx, B, H, W, kind, CO, CI):
    from synkrotomo_amd import _native as nat
    from synkrotomo_amd.projector import _ptr, _stream
    gen = torch.Generator(device="cuda").manual_seed(100 * kind + H)
    g = _ints(gen, (B, H, W, CO), -2, 2, torch.float32 if CO == 1 else torch.bfloat16)
    x = _ints(gen, (B, H, W, CI), -3, 3, torch.bfloat16 if CI == 32 else torch.float32)
    mask = None if kind == 2 else _ints(gen, (B, H, W, CO), -1, 1, torch.bfloat16)
    out = torch.empty(CO * 9 * CI + CO, device="cuda")
    nat.check(nat.lib().sk_conv_wgrad(ctx.handle, kind, B, H, W, _ptr(g), None if mask is None else _ptr(mask),
                                      _ptr(x), _ptr(out), _stream(ctx.device)), ctx.handle, "wgrad")
    gm = (g if mask is None else g * (mask > 0)).double().reshape(-1, CO)
    ref = torch.stack([gm.t() @ _shifted(x.double(), t).reshape(-1, CI) for t in range(9)], dim=1)  # [CO, 9, CI]
    assert torch.equal(out[:CO * 9 * CI].double(), ref.reshape(-1))
    assert torch.equal(out[CO * 9 * CI:].double(), gm.sum(0))


@pytest.mark.parametrize("B,H,W", SIZES)
@pytest.mark.parametrize("cin", [1, 2])
def test_first_layers_data_gradient_is_exact_on_integers(ctx, B, H, W, cin):
    from synkrotomo_amd import _native as nat
    from synkrotomo_amd.projector import _ptr, _stream
    L = nat.lib()
    gen = torch.Generator(device="cuda").manual_seed(10 * cin + W)
    dh = _ints(gen, (B, H, W, 32), -2, 2, torch.bfloat16)
    mask = _ints(gen, (B, H, W, 32), -1, 1, torch.bfloat16)
    w = _ints(gen, (32, 9, cin), -3, 3, torch.bfloat16)
    dx = torch.empty((B, H, W, cin), device="cuda")
    fn = L.sk_conv_in_dgrad if cin == 1 else L.sk_conv_in2_dgrad
    nat.check(fn(ctx.handle, B, H, W, _ptr(dh), _ptr(mask), _ptr(w), _ptr(dx), _stream(ctx.device)), ctx.handle,
              "dgrad")
    g1 = dh.double() * (mask > 0)
    ref = sum(_shifted(g1, 8 - t).reshape(-1, 32) @ w[:, t].double() for t in range(9))
    assert torch.equal(dx.double().reshape(-1, cin), ref)


@pytest.mark.parametrize("B,H,W", SIZES)
def test_masked_data_gradients_equal_masking_afterwards(ctx, B, H, W):
    """The gradients written with the ReLU derivative of the layer below are, bit for bit, the plain
    ones masked; and the first layer's from such a gradient is the one that masks it itself."""
    from synkrotomo_amd import _native as nat
    from synkrotomo_amd.projector import _ptr, _stream
    L, c, st = nat.lib(), ctx.handle, _stream(ctx.device)
    gen = torch.Generator(device="cuda").manual_seed(W)
    rnd = lambda *shape: torch.randn(shape, device="cuda", generator=gen)  # noqa: E731
    h = torch.relu(rnd(B, H, W, 32)).to(torch.bfloat16)
    zero = torch.zeros((), dtype=torch.bfloat16, device="cuda")
    g, w4 = rnd(B, H, W), rnd(9, 32).to(torch.bfloat16)
    a, b = torch.empty_like(h), torch.empty_like(h)
    nat.check(L.sk_conv_out_dgrad(c, B, H, W, _ptr(g), _ptr(w4), _ptr(a), st), c)
    nat.check(L.sk_conv_out_dgrad_relu(c, B, H, W, _ptr(g), _ptr(w4), _ptr(h), _ptr(b), st), c)
    assert torch.equal(torch.where(h > 0, a, zero), b)
    x, w = rnd(B, H, W, 32).to(torch.bfloat16), rnd(32, 9, 32).to(torch.bfloat16)
    wt = w.flip(1).permute(2, 1, 0).contiguous()
    nat.check(L.sk_conv32(c, B, H, W, _ptr(x), None, _ptr(wt), None, _ptr(a), st), c)
    nat.check(L.sk_conv32_dgrad_relu(c, B, H, W, _ptr(x), _ptr(w), _ptr(h), _ptr(b), st), c)
    assert torch.equal(torch.where(h > 0, a, zero), b)
    w1 = rnd(32, 9).to(torch.bfloat16)
    d0, d1 = torch.empty_like(g), torch.empty_like(g)
    nat.check(L.sk_conv_in_dgrad(c, B, H, W, _ptr(a), _ptr(h), _ptr(w1), _ptr(d0), st), c)
    nat.check(L.sk_conv_in_dgrad_relu(c, 1, B, H, W, _ptr(b), _ptr(w1), _ptr(d1), st), c)
    assert torch.equal(d0, d1)


# Sums that cancel to about 1e-6 of their terms: partials of two floats and FP64 sums keep 2^-40 of
# the terms, so the output is the FP64 sum rounded once (6e-8) or beside it (1.2e-7).
@pytest.mark.parametrize("B,H,W", [(1, 66, 66), (2, 17, 33), (5, 256, 256)])
def test_last_layers_bias_gradient_cancels_in_64_bits(ctx, B, H, W):
    from synkrotomo_amd import _native as nat
    from synkrotomo_amd.projector import _ptr, _stream
    g = torch.randn((B, H, W, 1), device="cuda", generator=torch.Generator(device="cuda").manual_seed(W))
    g.view(-1)[7] -= g.double().sum().float() + 1e-3
    x = torch.zeros((B, H, W, 32), device="cuda", dtype=torch.bfloat16)
    out = torch.empty(9 * 32 + 1, device="cuda")
    nat.check(nat.lib().sk_conv_wgrad(ctx.handle, 2, B, H, W, _ptr(g), None, _ptr(x), _ptr(out),
                                      _stream(ctx.device)), ctx.handle, "wgrad")
    want = g.double().sum().item()
    assert want != 0.0 and abs(out[-1].item() - want) <= 1.2e-7 * abs(want)
