"""Dense FP8 and MX GEMMs over the shapes where the choice between the split-K
strips, the 128x128 and the 256x256 kernels changes, with row remainders of
every tile height, K of one step up to more steps than a strip's ring holds,
K steps that do not divide by the waves, and every tile block of the 256x256
kernel (test_host_dense.py states which kernel takes which shape and that none is
left out).  +-1 operands (MX: exponents 2^-1, 1, 2 per 32-block): every partial
sum is a multiple of 1/4 below 2^17, exact in fp32 in any order, and the scales'
product is 2, so fp32 outputs must match a float64 product bit for bit and
bf16 outputs its rounding."""
import pytest
import torch

pytestmark = pytest.mark.gpu

SHAPES = [(1, 256, 128), (16, 256, 256), (17, 512, 1152), (31, 8192, 384), (33, 512, 384), (48, 256, 16384),
          (17, 8192, 2048), (64, 2048, 4224), (65, 2048, 1024), (130, 512, 4224), (129, 256, 2048),
          (300, 1024, 1152), (50, 16384, 256), (257, 4096, 4096), (1000, 1024, 2176), (63, 768, 640),
          (1000, 4096, 256), (777, 2048, 640), (2001, 2048, 384), (4095, 4096, 384), (300, 16384, 128),
          (1, 4352, 128), (16, 7168, 2048), (65, 32768, 1152), (12878, 1024, 1664), (32768, 512, 128),
          (65536, 256, 128), (200, 65536, 640)]


def _pm1(shape, gen):
    bits = torch.randint(0, 2, shape, generator=gen, device="cuda", dtype=torch.int32)
    return (bits * 2 - 1).to(torch.float32)


@pytest.mark.parametrize("mx", [False, True])
@pytest.mark.parametrize("m,n,k", SHAPES)
def test_dense_exact(hk, m, n, k, mx):
    gen = torch.Generator(device="cuda").manual_seed(m * 7 + n + k)
    a, b = _pm1((m, k), gen), _pm1((n, k), gen)
    a_q, b_q = a.to(torch.float8_e4m3fn), b.to(torch.float8_e4m3fn)
    a, b = a.double(), b.double()
    if mx:
        ea = torch.randint(126, 129, (m, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        eb = torch.randint(126, 129, (n, k // 32), generator=gen, device="cuda", dtype=torch.uint8)
        a = (a.view(m, -1, 32) * torch.exp2(ea.double() - 127)[..., None]).view(m, k)
        b = (b.view(n, -1, 32) * torch.exp2(eb.double() - 127)[..., None]).view(n, k)
        pa, pb = hk.mx_pack_scales(ea), hk.mx_pack_scales(eb)
    ref = a @ b.T if mx else 2.0 * (a @ b.T)
    sa, sb = torch.full((1,), 4.0, device="cuda"), torch.full((1,), 0.5, device="cuda")
    for dtype in (torch.float32, torch.bfloat16):
        # rows past the last one must stay untouched
        buf = torch.full((m + 1, n), 7.0, dtype=dtype, device="cuda")
        c = buf[:m]
        if mx:
            hk.tk_kernel.dispatch_gemm_mx(a_q, pa, b_q, pb, c)
        else:
            hk.tk_kernel.dispatch_gemm_fp8(a_q, b_q, c, sa, sb)
        torch.cuda.synchronize()
        assert torch.equal(c, ref.to(torch.float32).to(dtype))
        assert bool((buf[m] == 7.0).all())
        if not mx:  # each scale alone, and none
            for scales, factor in (((sa, None), 2.0), ((None, sb), 0.25), ((None, None), 0.5)):
                hk.tk_kernel.dispatch_gemm_fp8(a_q, b_q, c, *scales)
                torch.cuda.synchronize()
                assert torch.equal(c, (factor * ref).to(torch.float32).to(dtype)), scales
