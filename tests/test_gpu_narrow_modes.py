"""Narrow path of the one-call layers with per-tensor, block and MX scales: the
narrow kernels (64-row segments, and 16-row segments for at most 16 tokens) use
the 256x256 kernels' operand order, accumulation and epilogue, so a layer's
output is bit-identical with the narrow path on and off.  Shapes: K step counts
that are multiples of 8, of 4, odd, below the prefetch depth and above 64; token
counts on both sides of the 16-token and 64-token limits; both weight layouts; and,
with 256 experts, layers with experts of both kinds on both schedules (one stream,
and beside the 256x256 kernels with the late join)."""
import pytest
import torch

pytestmark = pytest.mark.gpu

#        H     I     E   k   (K steps: H / 128 and I / 128)
SHAPES = [(1024, 1024, 24, 4), (2304, 1152, 16, 4), (512, 1408, 12, 3), (256, 128, 8, 2), (256, 8320, 4, 2),
          (8448, 384, 4, 2), (512, 384, 256, 4)]


@pytest.fixture
def narrow_restore(hk):
    saved = hk.tk_kernel.get_narrow()
    yield
    hk.tk_kernel.set_narrow(*saved)


def _layer(hk, mode, H, I, E, k, packed, gen):
    w13 = torch.randn(E, 2 * I, H, device="cuda", generator=gen)
    w2 = torch.randn(E, H, I, device="cuda", generator=gen)
    if mode == "block":
        (a, sa), (b, sb) = hk.quant_block(w13), hk.quant_block(w2)
    elif mode == "mx":
        a, sa = hk.quant_mx(w13.view(E * 2 * I, H))
        b, sb = hk.quant_mx(w2.view(E * H, I))
        a, sa, b, sb = a.view(E, 2 * I, H), sa.view(E, 2 * I, -1), b.view(E, H, I), sb.view(E, H, -1)
    else:
        qa = [hk.quant_tensor(w13[e]) for e in range(E)]
        qb = [hk.quant_tensor(w2[e]) for e in range(E)]
        a, sa = torch.stack([q.view(torch.uint8) for q, _ in qa]).view(torch.float8_e4m3fn), torch.cat([s for _, s in qa])
        b, sb = torch.stack([q.view(torch.uint8) for q, _ in qb]).view(torch.float8_e4m3fn), torch.cat([s for _, s in qb])
    return (hk.MoELayerMX if mode == "mx" else hk.MoELayer)(a, sa, b, sb, k, pack=packed)


def _inputs(hk, mode, T, H, E, gen):
    x = torch.randn(T, H, device="cuda", generator=gen)
    logits = torch.randn(T, E, device="cuda", generator=gen)
    skew = 0.55 if E == 256 else 1.1
    logits -= skew * torch.log(torch.arange(1, E + 1, device="cuda").float())
    return {"block": hk.quant_group, "mx": hk.quant_mx, "tensor": hk.quant_tensor}[mode](x) + (logits,)


@pytest.mark.parametrize("packed", [True, False])
@pytest.mark.parametrize("mode", ["tensor", "block", "mx"])
@pytest.mark.parametrize("shape", SHAPES)
def test_narrow_matches_wide(hk, narrow_restore, mode, shape, packed):
    H, I, E, k = shape
    gen = torch.Generator(device="cuda").manual_seed(H + I + E)
    layer = _layer(hk, mode, H, I, E, k, packed, gen)
    # with 256 experts and weights in the packed layout, 65 tokens leave fewer small
    # experts than the mixed schedules ask for, 400 take them one after the other and
    # 11400 (178 rows per expert) MX and block scales on two streams
    for T in (1, 3, 16, 17, 64, 65, 150, 400) + ((11400,) if E == 256 else ()):
        args = _inputs(hk, mode, T, H, E, gen)
        hk.tk_kernel.set_narrow(0, 64, 0)
        off = layer(*args).clone()
        for setting in ((64, 64, 1), (64, 16, 2), (5, 64, 0)):
            hk.tk_kernel.set_narrow(*setting)
            on = layer(*args)
            torch.cuda.synchronize()
            assert torch.equal(on.view(torch.int16), off.view(torch.int16)), (T, setting)
        assert bool(torch.isfinite(off.float()).all())
        if E == 256 and T >= 400:  # experts of both kinds, enough small ones
            counts = torch.bincount(torch.topk(args[-1], k).indices.flatten(), minlength=E)
            assert bool((counts > 64).any()) and int(((counts > 0) & (counts <= 64)).sum()) >= 112


def test_mx_unaligned_exponents(hk):
    """Exponent bytes at an address that is not a multiple of 4 are refused."""
    gen = torch.Generator(device="cuda").manual_seed(5)
    layer = _layer(hk, "mx", 512, 256, 8, 2, True, gen)
    x_q, x_e, logits = _inputs(hk, "mx", 21, 512, 8, gen)
    flat = torch.empty(x_e.numel() + 1, dtype=torch.uint8, device="cuda")
    view = flat[1:].view(x_e.shape)
    view.copy_(x_e)
    with pytest.raises(RuntimeError, match="aligned"):
        layer(x_q, view, logits)
