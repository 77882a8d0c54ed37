"""Which kernels a layer call enqueues, on the host (no GPU): read from a stand-in
for the HIP runtime (fake_hip.cpp)."""
import json

import pytest

import hip_host


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return hip_host.build_fake(str(tmp_path_factory.mktemp("fake_hip")))


#          mode     T     E    H     I    packed  narrow GEMMs
LAYERS = [("tensor", 64, 256, 512, 256, 1, "alone"),    # every expert is narrow
          ("tensor", 65, 256, 256, 128, 1, "after"),    # all experts may turn out small
          ("mx", 2048, 220, 512, 256, 1, None),         # fewer experts
          ("mx", 2048, 256, 256, 128, 1, "after"),      # 64 rows per expert
          ("mx", 2049, 256, 256, 128, 1, None),         # above, 240 of 256 would have to be small
          ("mx", 8193, 1024, 256, 128, 1, "after"),     # 240 of 1024
          ("tensor", 2049, 256, 256, 128, 1, "after"),  # 111 of 256
          ("block", 2049, 256, 256, 128 * 3, 1, None),
          ("mx", 2049, 255, 4096, 1536, 1, None),
          ("mx", 2049, 256, 4096, 1536, 1, "after"),
          ("mx", 2049, 256, 4096, 1536, 0, None),       # row-major weights
          ("mx", 5632, 256, 4096, 1536, 1, "after"),    # 176 rows per expert
          ("mx", 5633, 256, 4096, 1536, 1, "beside"),
          ("mx", 5633, 256, 256, 128, 1, "beside"),
          ("block", 5633, 256, 4096, 1408, 1, "beside"),  # odd number of K steps
          ("tensor", 8192, 256, 4096, 1536, 1, "after"),  # 256
          ("tensor", 8193, 256, 4096, 1536, 1, None)]


@pytest.mark.parametrize("mode,T,E,H,I,packed,narrow", LAYERS)
def test_narrow_schedule(fake, mode, T, E, H, I, packed, narrow):
    call = {"tensor": "moe(T, E, 8, H, I, TENSOR, packed, 1001)", "block": "moe(T, E, 8, H, I, BLOCK, packed, 1001)",
            "mx": "moe_mx(T, E, 8, H, I, packed, 1001)"}[mode]
    out = hip_host.run(fake, f"""
    T, E, H, I, packed = {T}, {E}, {H}, {I}, {packed}
    assert {call} == 0, lib.hkmoe_last_error()
    print(json.dumps([x for x in log() if "gemm_fp8" in x]))
    """)
    gemms = ["narrow" if "gemm_fp8_narrow" in x else "wide" for x in json.loads(out[-1])]
    streams = {x.rsplit("=", 1)[1] for x in json.loads(out[-1])}
    assert gemms == {None: ["wide"] * 2, "alone": ["narrow"] * 2, "after": ["wide", "narrow"] * 2,
                     "beside": ["narrow"] * 2 + ["wide"] * 2}[narrow]
    assert len(streams) == (2 if narrow == "beside" else 1)
