"""Which kernel a dense GEMM call launches, on the host (no GPU): read from a stand-in
for the HIP runtime (fake_hip.cpp)."""
import json
import re

import pytest

import hip_host
import test_gpu_dense_shapes
import test_gpu_gemm


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return hip_host.build_fake(str(tmp_path_factory.mktemp("fake_hip")))


def launches(fake, calls, mfma):
    """The launch line of each (m, n, k, f32, mx)."""
    out = hip_host.run(fake, f"""
    assert lib.hkmoe_set_dense_mfma({mfma}) == 0
    for c in {calls!r}:
        assert dense(*c) == 0, lib.hkmoe_last_error()
    print(json.dumps(log()))
    """)
    lines = json.loads(out[-1])
    assert len(lines) == len(calls)
    return lines


def kernels(fake, calls, mfma=32):
    """The kernel of each call: "strip MFxNF" (16 MF rows, 16 NF columns), "128" or "256"."""
    names = []
    for line in launches(fake, calls, mfma):
        m = re.match(r"launch hkmoe::gemm_fp8_(skinny<(\d), *_?(\d), *_?(\d)|small|persistent)", line)
        names.append(f"strip {m.group(2)}x{m.group(3)}" if m.group(2) else {"small": "128", "persistent": "256"}[m.group(1)])
    return names


# m, n, k, f32, mx and the kernel that takes them (times in us, 128x128 tiles first)
PICKS = [((2048, 2048, 2048, 0, 0), "128"), ((8192, 8192, 2048, 0, 0), "256"), ((17, 8192, 2048, 0, 0), "strip 2x2"),
         ((8192, 8192, 8192, 1, 1), "256"), ((4096, 4096, 4096, 0, 0), "256"),
         # the last of several rounds of 256x256 tiles is nearly empty: 38.2 / 35.5
         ((6000, 3072, 1024, 0, 1), "256"), ((6000, 3072, 2048, 0, 1), "256"), ((12000, 1536, 512, 0, 1), "256"),
         # one row of 128x128 tiles, on two rounds of the CUs that it gets: 24.5 / 16.3 in strips
         ((65, 11264, 2048, 1, 1), "strip 4x4"), ((96, 11264, 2048, 1, 0), "strip 4x4"),
         ((200, 6144, 4096, 0, 0), "128"),  # two rows of tiles, one round: 19.7 / 25.0
         # one K step, fp32 output: 13.4 / 16.9
         ((12000, 768, 128, 1, 1), "128"), ((6000, 1536, 128, 1, 0), "128")]


def test_picks(fake):
    assert kernels(fake, [c for c, _ in PICKS]) == [k for _, k in PICKS]


def test_gpu_shapes_reach_every_kernel(fake):
    """Every form of every dense kernel has a shape in the GPU test, and the 256x256
    kernel each of its tile blocks (2^b M tiles x 2^(5-b) N tiles)."""
    want = {"strip 1x1", "strip 2x1", "strip 1x2", "strip 2x2", "strip 2x4", "strip 4x4", "128", "256"}
    for mx in (0, 1):
        for f32 in (0, 1):
            got = kernels(fake, [(m, n, k, f32, mx) for m, n, k in test_gpu_dense_shapes.SHAPES])
            assert set(got) == want, (mx, f32, want - set(got))
            blocks = set()
            for (m, n, _), kern in zip(test_gpu_dense_shapes.SHAPES, got):
                mt, nt = -(-m // 256), n // 256
                rounds = lambda b: -(-(-(-mt // 2 ** b) * -(-nt // 2 ** (5 - b))) // 8)
                if kern == "256":
                    blocks.add(min((2, 3, 1, 4, 5, 0), key=rounds))
            assert blocks >= {0, 2, 3, 4, 5} | ({1} if f32 == 0 else set()), blocks


def test_mfma_shapes_of_the_128_kernel(fake):
    """The GPU test's shapes of the 128x128 kernel run on it, on the MFMA asked for
    (template arguments: fp32 output, 32x32x64, MX)."""
    for mfma in (16, 32):
        for f32 in (0, 1):
            calls = [(m, n, k, f32, 0) for m, n, k in test_gpu_gemm.SMALL_KERNEL]
            form = f"gemm_fp8_small<{'true' if f32 else 'false'},_{'true' if mfma == 32 else 'false'},_false>"
            for c, line in zip(calls, launches(fake, calls, mfma)):
                assert form in line, (c, line)
