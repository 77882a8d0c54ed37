"""Which kernel a dense GEMM call launches, on the host (no GPU): read from a stand-in
for the HIP runtime (fake_hip.cpp)."""
import json
import re

import pytest

import hip_host


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return hip_host.build_fake(str(tmp_path_factory.mktemp("fake_hip")))


def kernels(fake, calls, mfma=32):
    """The kernel of each (m, n, k, f32, mx): "strip <MF, NF, NW>", "128" or "256"."""
    out = hip_host.run(fake, f"""
    assert lib.hkmoe_set_dense_mfma({mfma}) == 0
    for c in {calls!r}:
        assert dense(*c) == 0, lib.hkmoe_last_error()
    print(json.dumps(log()))
    """)
    names = []
    for line in json.loads(out[-1]):
        m = re.match(r"launch hkmoe::gemm_fp8_(skinny<(\d), *_?(\d), *_?(\d)|small|persistent)", line)
        names.append(f"strip {m.group(2)}x{m.group(3)}" if m.group(2) else {"small": "128", "persistent": "256"}[m.group(1)])
    assert len(names) == len(calls)
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
