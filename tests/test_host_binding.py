"""The pybind11 module on the host (no GPU): tk_kernel over a stand-in for the HIP
runtime (fake_hip.cpp) and a stand-in for torch."""
import pytest

import hip_host


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return hip_host.build_fake(str(tmp_path_factory.mktemp("fake_hip")))


@pytest.mark.parametrize("ndim", [0, 1, 2, 7, 8, 9, 10, 17, 40])
def test_quant_tensor_of_any_rank(fake, ndim):
    """The per-tensor quantiser takes a tensor of any rank; sizes past the
    inline ones count (1 x ... x 1 x 3 x 5 values, 15 of q and not 14)."""
    shape = ([1] * ndim + [3, 5])[-ndim:] if ndim else []
    out = hip_host.run(fake, hip_host.BINDING + f"""
shape, f8 = {shape!r}, "torch.float8_e4m3fn"
one = Tensor([1])
tk_kernel.dispatch_quant_tensor(Tensor(shape), Tensor(shape, f8), one, one)
print(log())
try:
    tk_kernel.dispatch_quant_tensor(Tensor(shape), Tensor([14], f8), one, one)
except RuntimeError as e:
    print(e)
""")
    assert "quant_tensor_small_kernel" in out[-2] and "stream=7" in out[-2]
    assert "q like x" in out[-1]
