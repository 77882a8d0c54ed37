"""Device quantisers at the edges of their tilings: partial workgroups, odd
value counts, both sides of the per-tensor one-launch limit (2^17 values),
unaligned views, and NaN / infinity, against the CPU specification (bit-exact)."""
import numpy as np
import pytest
import torch

from helpers import f8_np
from oracle import mx, spec

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def tk():
    import hkmoe
    return hkmoe.tk_kernel


def _data(shape, seed):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal(shape).astype(np.float32)
    x *= np.float32(2.0) ** rng.integers(-12, 12, shape[:-1] + (1,)).astype(np.float32)
    x.reshape(-1)[: 3] = [-0.0, 0.0, 1e-30][: min(3, x.size)]
    return x


def _at(arr, off, dtype):
    """arr on the GPU at a storage offset of `off` elements (a contiguous view)."""
    flat = torch.empty(arr.size + off, dtype=dtype, device="cuda")
    flat[off:].copy_(torch.from_numpy(arr.reshape(-1)))
    return flat[off:].view(arr.shape)


def _out(shape, off):
    n = int(np.prod(shape))
    return torch.empty(n + off, dtype=torch.uint8, device="cuda")[off:].view(torch.float8_e4m3fn).view(shape)


CASES = [("group", (1, 128)), ("group", (31, 128)), ("group", (5, 7168)), ("group", (133, 384)),
         ("block", (1, 128, 128)), ("block", (3, 256, 384)),
         ("tensor", (1, 1)), ("tensor", (3, 1)), ("tensor", (29, 4096)), ("tensor", (1, 131072)),
         ("tensor", (1, 131073)), ("tensor", (301, 4099)), ("tensor", (2050, 4096))]


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("what,shape", CASES)
def test_quantiser_edges(tk, what, shape, off):
    x = _data(shape, seed=sum(shape) + off)
    ref = {"group": spec.quant_group_1x128, "block": spec.quant_block_128x128, "tensor": spec.quant_per_tensor}[what]
    q_ref, s_ref = ref(x)
    s_ref = np.atleast_1d(np.asarray(s_ref, np.float32))
    xg, q = _at(x, off, torch.float32), _out(shape, off)
    s = torch.empty(s_ref.shape, dtype=torch.float32, device="cuda")
    if what == "tensor":
        tk.dispatch_quant_tensor(xg, q, s, torch.empty(1, dtype=torch.float32, device="cuda"))
    else:
        (tk.dispatch_quant_group if what == "group" else tk.dispatch_quant_block)(xg, q, s)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(f8_np(q).reshape(shape), q_ref.reshape(shape))
    np.testing.assert_array_equal(s.cpu().numpy(), s_ref)


@pytest.mark.parametrize("what,shape", [("group", (6, 256)), ("block", (1, 256, 256)), ("tensor", (6, 256)),
                                        ("tensor", (64, 4096))])
def test_quantiser_non_finite(tk, what, shape):
    """NaNs do not enter the scale and give the NaN code; an infinite maximum
    gives an infinite scale, zeros for finite values and the NaN code for inf / inf."""
    x = _data(shape, seed=1)
    flat = x.reshape(-1)
    clean = x.copy()
    flat[7], clean.reshape(-1)[7] = np.nan, 0.0
    ref = {"group": spec.quant_group_1x128, "block": spec.quant_block_128x128, "tensor": spec.quant_per_tensor}[what]
    for inf in (False, True):
        if inf:
            flat[64] = -np.inf
        q = _out(shape, 0)
        q_ref, s_ref = ref(clean)
        s_ref = np.atleast_1d(np.asarray(s_ref, np.float32))
        s = torch.empty(s_ref.shape, dtype=torch.float32, device="cuda")
        xg = torch.from_numpy(x).cuda()
        if what == "tensor":
            tk.dispatch_quant_tensor(xg, q, s, torch.empty(1, dtype=torch.float32, device="cuda"))
        else:
            (tk.dispatch_quant_group if what == "group" else tk.dispatch_quant_block)(xg, q, s)
        torch.cuda.synchronize()
        got, s = f8_np(q).reshape(-1), s.cpu().numpy().reshape(-1)
        q_ref = q_ref.reshape(-1).copy()
        if inf:  # everything that shares the infinite scale
            share = np.zeros(shape, bool)
            (share.reshape(shape[0], -1, 128)[:1, :1] if what == "group" else
             share[:, :128, :128] if what == "block" else share)[...] = True
            q_ref = np.where(share.reshape(-1), np.where(np.signbit(clean.reshape(-1)), 0x80, 0), q_ref).astype(np.uint8)
            assert np.isinf(s[0])
            np.testing.assert_array_equal(s[1:], s_ref.reshape(-1)[1:])
            assert got[64] & 0x7F == 0x7F
            q_ref[64] = got[64]
        else:
            np.testing.assert_array_equal(s, s_ref.reshape(-1))
        assert got[7] & 0x7F == 0x7F
        q_ref[7] = got[7]
        np.testing.assert_array_equal(got, q_ref)


@pytest.mark.parametrize("off", [0, 1])
@pytest.mark.parametrize("rows,cols", [(1, 32), (63, 32), (64, 32), (65, 32), (127, 160), (2048, 4096), (2049, 4096)])
def test_quant_mx_edges(tk, rows, cols, off):
    """MX: partial workgroups and both sides of the two kernels' line (2^23 values)."""
    x = _data((rows, cols), seed=rows + off)
    q_ref, s_ref = mx.quant_mx(x)
    # what lies around the outputs must stay untouched
    q_buf = torch.full((rows * cols + off + 64,), 0x55, dtype=torch.uint8, device="cuda")
    s_buf = torch.full((rows * cols // 32 + 64,), 0x55, dtype=torch.uint8, device="cuda")
    q = q_buf[off:off + rows * cols].view(torch.float8_e4m3fn).view(rows, cols)
    s = s_buf[:rows * cols // 32].view(rows, cols // 32)
    tk.dispatch_quant_mx(_at(x, off, torch.float32), q, s)
    torch.cuda.synchronize()
    np.testing.assert_array_equal(f8_np(q), q_ref)
    np.testing.assert_array_equal(s.cpu().numpy(), s_ref)
    assert bool((q_buf[:off] == 0x55).all()) and bool((q_buf[off + rows * cols:] == 0x55).all())
    assert bool((s_buf[rows * cols // 32:] == 0x55).all())
