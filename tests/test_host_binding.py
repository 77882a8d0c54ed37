"""The pybind11 module on the host (no GPU): tk_kernel over a stand-in for the HIP
runtime (fake_hip.cpp) and a stand-in for torch."""
import subprocess

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


def test_first_calls_of_two_threads_do_not_deadlock(fake):
    """The binding looks torch up on its first call.  That runs Python code,
    which may hand the GIL to a second thread that makes its own first call."""
    try:
        out = hip_host.run(fake, hip_host.BINDING + """
real = builtins.__import__
def slow(name, *a, **kw):
    if name == "torch":
        time.sleep(0.5)  # the GIL goes to the other thread
    return real(name, *a, **kw)
builtins.__import__ = slow
one, done = Tensor([1]), []
def work():
    tk_kernel.dispatch_quant_tensor(Tensor([4]), Tensor([4], "torch.float8_e4m3fn"), one, one)
    done.append(1)
ts = [threading.Thread(target=work) for _ in range(3)]
[t.start() for t in ts]
[t.join() for t in ts]
print(len(done), sum("quant_tensor_small_kernel" in x for x in log()))
""", timeout=30)
    except subprocess.TimeoutExpired:
        pytest.fail("the threads' first calls wait for each other")
    assert out[-1] == "3 3"
