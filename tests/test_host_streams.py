"""The auxiliary stream of the one-call layers, on the host (no GPU): which
streams and events the library creates and in which order it enqueues on them,
read from a stand-in for the HIP runtime (fake_hip.cpp)."""
import json
import re

import pytest

import hip_host


@pytest.fixture(scope="module")
def fake(tmp_path_factory):
    return hip_host.build_fake(str(tmp_path_factory.mktemp("fake_hip")))


CALL = {"block": "moe(8192, 64, 4, 512, 256, BLOCK, 1, s)", "mx": "moe_mx(16384, 256, 4, 4096, 1536, 1, s)"}


@pytest.mark.parametrize("call", list(CALL.values()), ids=list(CALL))
def test_first_calls_of_two_threads_share_one_stream(fake, call):
    """Two host threads whose first layer calls overlap: one auxiliary stream and
    one pair of events, and every wait is for an event that was recorded before."""
    out = hip_host.run(fake, f"""
    hip.fake_hip_delay(200)
    gate, rcs = threading.Barrier(2), [None, None]
    def work(n):
        s = 1001 + n
        gate.wait()
        rcs[n] = {call}
    ts = [threading.Thread(target=work, args=(n,)) for n in range(2)]
    [t.start() for t in ts]
    [t.join() for t in ts]
    print(json.dumps([rcs, log()]))
    """)
    rcs, lines = json.loads(out[-1])
    assert rcs == [0, 0]
    assert sum(x.startswith("stream_create") for x in lines) == 1, lines
    assert sum(x.startswith("event_create") for x in lines) == 2, lines
    aux = re.search(r"stream_create (\d+)", "\n".join(lines)).group(1)
    recorded, forks = {}, 0
    for x in lines:
        m = re.match(r"(record|wait) (\d+) stream=(\d+)", x)
        if not m:
            continue
        what, event, stream = m.groups()
        if what == "record":
            recorded[event] = stream
        else:
            # the auxiliary stream waits for a caller's stream and the other way round
            assert event in recorded and (recorded[event] == aux) != (stream == aux), lines
            forks += stream == aux
    assert forks == 2
    # one thread's whole fork / join is enqueued before the other's starts
    order = [m.group(1) for m in (re.search(r"^(?:record|wait) .* ?stream=(100\d)", x) for x in lines) if m]
    assert order in (["1001"] * 2 + ["1002"] * 2, ["1002"] * 2 + ["1001"] * 2), lines


@pytest.mark.parametrize("fn,after", [("hipStreamCreateWithFlags", 0), ("hipEventCreateWithFlags", 0),
                                      ("hipEventCreateWithFlags", 1)])
def test_failed_creation_leaves_nothing_behind(fake, fn, after):
    """A stream or event that cannot be created fails the call, what had been
    created is destroyed, and the next call starts afresh."""
    out = hip_host.run(fake, f"""
    s = 1001
    hip.fake_hip_fail(b"{fn}", {after})
    rc = {CALL["block"]}
    print(json.dumps([rc, lib.hkmoe_last_error().decode(), log()]))
    rc = {CALL["block"]}
    print(json.dumps([rc, "", log()]))
    """)
    (rc, err, lines), (rc2, _, lines2) = [json.loads(x) for x in out[-2:]]
    assert rc == 3 and "auxiliary" in err
    assert not any(x.startswith("launch") for x in lines)
    made = [x.split()[1] for x in lines if "_create" in x]
    gone = [x.split()[1] for x in lines if "_destroy" in x]
    assert sorted(made) == sorted(gone), lines
    assert rc2 == 0
    assert sum("_create" in x for x in lines2) == 3 and sum(x.startswith("launch") for x in lines2) >= 8


def test_no_creation_under_capture(fake):
    """A first call under capture creates nothing and runs on the caller's stream;
    the lock is free again for the next one."""
    out = hip_host.run(fake, f"""
    s = 1001
    hip.fake_hip_capturing(1)
    for _ in range(2):
        assert {CALL["block"]} == 0
        print(json.dumps(log()))
    hip.fake_hip_capturing(0)
    assert {CALL["block"]} == 0
    print(json.dumps(log()))
    """)
    first, second, third = [json.loads(x) for x in out[-3:]]
    assert first == second and not any("_create" in x or "wait" in x for x in first)
    assert all(x.endswith("stream=1001") for x in first if x.startswith("launch"))
    assert sum("_create" in x for x in third) == 3
