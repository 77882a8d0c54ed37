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
    # with 256 experts, weights in the packed layout and at most 64 tokens per-tensor and
    # MX layers take the narrow kernels, with more only where no expert is larger (these
    # layers are too small for both kinds, see below); block scales at every T, at
    # 11400 (178 rows per expert) on two streams
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
        if E == 256 and T >= 400:  # experts of both kinds
            counts = torch.bincount(torch.topk(args[-1], k).indices.flatten(), minlength=E)
            assert bool((counts > 64).any()) and int(((counts > 0) & (counts <= 64)).sum()) >= 112


def _narrow_count(hk, layer, T):
    """Narrow experts of the last call: after the routing tables in the workspace."""
    E, r, nblk = layer.num_experts, T * layer.top_k, hk.tk_kernel.route_blocks(T)
    sizes = [r, r, nblk * E, nblk * E, E, E + 1, E + 1, 2 * ((r + 255) // 256 + E), 1, 16]
    at = sum((4 * n + 255) // 256 * 256 for n in sizes)
    return int(layer._ws[at:at + 4].view(torch.int32))


def _pays(small, H, I, mode):
    """The narrow kernels take these experts (their row counts) beside larger ones
    on one stream."""
    mb = 3e-6 * H * I
    need, per_expert, per_row = (40000, 360 + 6 * mb, 0.6 * mb) if mode == "tensor" else (60000, 250 + 15 * mb, 2 + 0.4 * mb)
    return len(small) * int(per_expert + 0.5) - int(small.sum()) * int(per_row + 0.5) >= need


@pytest.mark.parametrize("mode", ["tensor", "mx"])
@pytest.mark.parametrize("E,T,hot", [(256, 200, False), (256, 200, True), (256, 1200, True), (1024, 1000, False),
                                     (1024, 1000, True), (1024, 7500, True), (1024, 8200, True)])
def test_which_experts_are_narrow(hk, narrow_restore, mode, E, T, hot):
    """Small layers, on one stream: with no larger expert all are narrow, beside larger
    ones they are if enough of them of few enough rows are there, on average above 64
    rows per expert too."""
    H, I, k = 256, 128, 8
    gen = torch.Generator(device="cuda").manual_seed(E + T)
    layer = _layer(hk, mode, H, I, E, k, True, gen)
    x = torch.randn(T, H, device="cuda", generator=gen)
    logits = torch.randn(T, E, device="cuda", generator=gen)
    if T > 8000:  # half of the experts take most tokens
        logits[:, ::2] += 1.0
    logits[:, 7] += 30.0 if hot else 0.0
    if (E, T) == (256, 200) and hot:  # and the rest goes to the first 100
        logits[:, :100] += 20.0
    args = (hk.quant_mx if mode == "mx" else hk.quant_tensor)(x) + (logits,)
    out = layer(*args).clone()
    got = _narrow_count(hk, layer, T)
    hk.tk_kernel.set_narrow(0, 64, 0)
    off = layer(*args)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), off.view(torch.int16))
    counts = torch.bincount(torch.topk(logits, k, dim=1)[1].flatten(), minlength=E)
    small = counts[(counts > 0) & (counts <= 64)]
    assert bool((counts > 64).any()) == hot
    pays = _pays(small, H, I, mode)
    assert pays == ((E, T) in ((1024, 1000), (1024, 7500), (1024, 8200)) or (mode, E, T) == ("tensor", 256, 1200) or not hot)
    assert got == (len(small) if not hot or pays else 0)


def _codes(gen, *shape):
    """Random e4m3 bytes of magnitude 2^-3 .. 2^1, both signs."""
    b = torch.randint(0, 256, shape, generator=gen, device="cuda", dtype=torch.uint8)
    return ((b & 0x9f) | 0x20).view(torch.float8_e4m3fn)


def _large_layer(hk, mode):
    """256 experts of 25 MB (block: 27 MB and an odd number of K steps)."""
    E, H, I, k = 256, 4096, 2176 if mode == "block" else 2048, 8
    gen = torch.Generator(device="cuda").manual_seed(I)
    w13, w2 = _codes(gen, E, 2 * I, H), _codes(gen, E, H, I)
    if mode == "mx":
        s13, s2 = (torch.randint(115, 119, (E, n, c // 32), generator=gen, device="cuda", dtype=torch.uint8)
                   for n, c in ((2 * I, H), (H, I)))
        return hk.MoELayerMX(w13, s13, w2, s2, k)
    s13, s2 = (torch.rand((E,) if mode == "tensor" else (E, n // 128, c // 128), generator=gen, device="cuda") * 0.004
               for n, c in ((2 * I, H), (H, I)))
    return hk.MoELayer(w13, s13, w2, s2, k)


def _large_inputs(hk, layer, mode, T, seed):
    """24 experts of many rows, some 200 of few."""
    gen = torch.Generator(device="cuda").manual_seed(seed)
    logits = torch.randn(T, layer.num_experts, device="cuda", generator=gen)
    logits[:, :24] += 2.6
    x = torch.randn(T, layer.hidden, device="cuda", generator=gen)
    return {"block": hk.quant_group, "mx": hk.quant_mx, "tensor": hk.quant_tensor}[mode](x) + (logits,)


@pytest.mark.parametrize("mode", ["tensor", "block", "mx"])
def test_both_kinds_of_experts(hk, narrow_restore, mode):
    """Narrow kernels beside the 256x256 ones where the small experts pay for them:
    one after the other, and (6500 tokens, block and MX scales) on two streams."""
    layer = _large_layer(hk, mode)
    for T in (2000, 6500):
        args = _large_inputs(hk, layer, mode, T, T)
        counts = torch.bincount(torch.topk(args[-1], layer.top_k, dim=1)[1].flatten(), minlength=layer.num_experts)
        small = counts[(counts > 0) & (counts <= 64)]
        assert _pays(small, layer.hidden, layer.inter, mode) and bool((counts > 256).any())
        out = layer(*args).clone()
        assert _narrow_count(hk, layer, T) == len(small)
        hk.tk_kernel.set_narrow(0, 64, 0)
        off = layer(*args).clone()
        hk.tk_kernel.set_narrow(64, 64, 2)
        join = layer(*args)
        hk.tk_kernel.set_narrow(64, 64, 1)
        torch.cuda.synchronize()
        assert bool(torch.isfinite(off.float()).all())
        assert torch.equal(out.view(torch.int16), off.view(torch.int16))
        assert torch.equal(join.view(torch.int16), off.view(torch.int16))


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
