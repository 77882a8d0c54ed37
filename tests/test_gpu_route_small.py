"""Routing of at most 64 tokens (one launch inside the one-call layers) against
the three-launch routing that larger batches and the stepwise layer use: same top-k,
row order and weights, so the same output bits, at the edges of its token, expert and
top-k ranges, with ties in the logits."""
import pytest
import torch

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("T", [1, 2, 31, 33, 63, 64])
@pytest.mark.parametrize("E,k", [(1, 1), (16, 16), (17, 3), (40, 32), (129, 8), (1024, 32)])
def test_small_routing_matches_steps(hk, T, E, k):
    H, I = 256, 128
    gen = torch.Generator(device="cuda").manual_seed(T * 1000 + E)
    w13_q, w13_s = hk.quant_block(torch.randn(E, 2 * I, H, device="cuda", generator=gen))
    w2_q, w2_s = hk.quant_block(torch.randn(E, H, I, device="cuda", generator=gen))
    x_q, x_s = hk.quant_group(torch.randn(T, H, device="cuda", generator=gen))
    logits = torch.randn(T, E, device="cuda", generator=gen)
    logits[T // 2] = torch.round(logits[T // 2])  # many ties in one row
    steps = hk.moe_forward_steps(x_q, x_s, logits, w13_q, w13_s, w2_q, w2_s, k)
    out = hk.moe_forward(x_q, x_s, logits, w13_q, w13_s, w2_q, w2_s, k)
    again = hk.moe_forward(x_q, x_s, logits, w13_q, w13_s, w2_q, w2_s, k)
    torch.cuda.synchronize()
    assert torch.equal(out.view(torch.int16), steps["out"].view(torch.int16))
    assert torch.equal(out.view(torch.int16), again.view(torch.int16))


@pytest.mark.parametrize("E,k", [(16, 16), (40, 12), (300, 32)])
def test_topk_order_of_special_logits(hk, E, k):
    """Descending order with ties (-0 and +0 among them) to the lower expert id;
    -inf below every number and NaN below -inf."""
    gen = torch.Generator().manual_seed(E)
    logits = torch.round(torch.randn(40, E, generator=gen) * 2)
    pick = torch.randint(0, 6, (40, E), generator=gen)
    logits[pick == 0] = float("-inf")
    logits[(pick == 1) & (logits == 0)] = -0.0
    logits[1::2][pick[1::2] == 2] = float("nan")
    logits[3, : E // 2] = float("inf")
    logits[5] = float("nan")
    rank = torch.where(logits.isnan(), torch.tensor(float("-inf")), logits)
    # sorted is stable: NaN last, value descending, then id
    want = torch.tensor([sorted(range(E), key=lambda e: (bool(row[e].isnan()), -float(r[e])))[:k]
                         for row, r in zip(logits, rank)], dtype=torch.int32)
    idx = torch.empty((40, k), dtype=torch.int32, device="cuda")
    w = torch.empty((40, k), dtype=torch.float32, device="cuda")
    bc = torch.empty((hk.tk_kernel.route_blocks(40), E), dtype=torch.int32, device="cuda")
    hk.tk_kernel.dispatch_route_topk(logits.cuda(), idx, w, bc)
    torch.cuda.synchronize()
    assert torch.equal(idx.cpu(), want)
    assert int(bc.sum()) == 40 * k


@pytest.mark.parametrize("T", [24, 64, 65, 100])
@pytest.mark.parametrize("hot", [True, False])
def test_narrow_experts_of_few_tokens(hk, T, hot):
    """MX layer of 256 experts with packed weights and the narrow limit at 16 rows.
    A few small experts beside one that every token takes are not enough for the
    narrow kernels, some 130 and more without a larger one are, whether routing is one
    launch (T <= 64) or three."""
    E, H, I, k = 256, 256, 128, 2 if hot else 8
    gen = torch.Generator(device="cuda").manual_seed(T + k)
    w13_q, w13_e = hk.quant_mx(torch.randn(E * 2 * I, H, device="cuda", generator=gen))
    w2_q, w2_e = hk.quant_mx(torch.randn(E * H, I, device="cuda", generator=gen))
    layer = hk.MoELayerMX(w13_q.view(E, 2 * I, H), w13_e.view(E, 2 * I, -1), w2_q.view(E, H, I), w2_e.view(E, H, -1), k)
    x_q, x_e = hk.quant_mx(torch.randn(T, H, device="cuda", generator=gen))
    logits = torch.randn(T, E, device="cuda", generator=gen)
    logits[:, 7] += 30.0 if hot else 0.0
    saved = hk.tk_kernel.get_narrow()
    hk.tk_kernel.set_narrow(64, 16, 1)
    try:
        layer(x_q, x_e, logits)
        torch.cuda.synchronize()
    finally:
        hk.tk_kernel.set_narrow(*saved)
    counts = torch.bincount(torch.topk(logits, k, dim=1)[1].flatten(), minlength=E)
    small = int(((counts > 0) & (counts <= 16)).sum())
    assert bool((counts > 16).any()) == hot and (0 < small < 112) == hot
    # the count of narrow experts, after the routing tables in the workspace
    r, nblk = T * k, hk.tk_kernel.route_blocks(T)
    sizes = [r, r, nblk * E, nblk * E, E, E + 1, E + 1, 2 * ((r + 255) // 256 + E), 1, 16]
    at = sum((4 * n + 255) // 256 * 256 for n in sizes)
    assert int(layer.workspace(T, "cuda")[at:at + 4].view(torch.int32)) == (0 if hot else small)
