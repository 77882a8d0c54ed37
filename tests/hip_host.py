"""Runs a snippet against libhkmoe.so with the HIP runtime of fake_hip.cpp in
place of the real one (a child process; no GPU, nothing is launched)."""
import os
import subprocess
import sys
import textwrap

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))
LIB = os.path.join(ROOT, "distributed-hipkittens_amd", "libhkmoe.so")

PRELUDE = f"""
import ctypes, json, sys, threading
hip = ctypes.CDLL("libamdhip64.so.7", mode=ctypes.RTLD_GLOBAL)
lib = ctypes.CDLL({LIB!r})
hip.fake_hip_log.restype = ctypes.c_char_p
lib.hkmoe_last_error.restype = ctypes.c_char_p
lib.hkmoe_moe_workspace_size.restype = ctypes.c_size_t
i32, i64, vp = ctypes.c_int32, ctypes.c_int64, ctypes.c_void_p
P = vp(1 << 20)  # stands for every device buffer: never dereferenced
TENSOR, BLOCK = 0, 1

def log():
    lines = hip.fake_hip_log().decode().split("\\n")[:-1]
    hip.fake_hip_clear()
    return lines

def moe(T, E, k, H, I, mode, packed, stream):
    return lib.hkmoe_moe_forward(P, P, P, P, P, P, P, i64(T), i32(E), i32(k), i32(H), i32(I), mode, packed, P, P,
                                 ctypes.c_size_t(1 << 50), vp(stream))

def moe_mx(T, E, k, H, I, packed, stream):
    return lib.hkmoe_moe_forward_mx(P, P, P, P, P, P, P, i64(T), i32(E), i32(k), i32(H), i32(I), packed, P, P,
                                    ctypes.c_size_t(1 << 50), vp(stream))

def dense(m, n, k, f32, mx):
    if mx:
        return lib.hkmoe_gemm_mx(P, P, P, P, P, i64(m), i64(n), i64(k), int(f32), None)
    return lib.hkmoe_gemm_fp8(P, P, P, i64(m), i64(n), i64(k), P, P, int(f32), None)
"""


def build_fake(directory):
    """libamdhip64.so.7 in `directory`."""
    so = os.path.join(directory, "libamdhip64.so.7")
    versions = os.path.join(directory, "hip.map")
    with open(versions, "w") as f:  # the versions that libhkmoe.so asks for
        f.write("hip_4.2 { global: *; };\nhip_4.3 { global: hipStreamIsCapturing; } hip_4.2;\n")
    subprocess.run(["g++", "-O1", "-g", "-std=c++17", "-fPIC", "-shared", "-pthread",
                    "-Wl,-soname,libamdhip64.so.7", f"-Wl,--version-script={versions}",
                    os.path.join(ROOT, "tests", "fake_hip.cpp"), "-o", so], check=True, capture_output=True, text=True)
    return directory


def run(fake_dir, snippet, timeout=60):
    """stdout lines of the snippet (it sees PRELUDE's names)."""
    env = dict(os.environ, LD_LIBRARY_PATH=":".join([fake_dir] + os.environ.get("LD_LIBRARY_PATH", "").split(":")).rstrip(":"))
    for name in ("HKMOE_NARROW_CUS", "HKMOE_NARROW_MAX", "HKMOE_NARROW_SHARE"):
        env.pop(name, None)
    res = subprocess.run([sys.executable, "-c", PRELUDE + textwrap.dedent(snippet)], capture_output=True, text=True,
                         env=env, timeout=timeout)
    assert res.returncode == 0, res.stdout[-3000:] + res.stderr[-3000:]
    return res.stdout.split("\n")[:-1]


# tk_kernel over the stand-in runtime: torch is a stand-in too (the real one would
# load its own HIP libraries), Tensor a class with the attributes the binding reads.
BINDING = f"""
import builtins, sys, time, types
torch = types.ModuleType("torch")
class Tensor:
    def __init__(self, shape, dtype="torch.float32", device="cuda"):
        self.shape, self.dtype, self.device = tuple(shape), dtype, types.SimpleNamespace(type=device)
        self.is_cpu = device == "cpu"
    def is_contiguous(self):
        return True
    def data_ptr(self):
        return 1 << 20
torch.Tensor, torch._C = Tensor, types.SimpleNamespace()
torch.cuda = types.SimpleNamespace(current_stream=lambda: types.SimpleNamespace(cuda_stream=7))
sys.modules["torch"] = torch
sys.path.insert(0, {os.path.dirname(LIB)!r})
import tk_kernel
"""
