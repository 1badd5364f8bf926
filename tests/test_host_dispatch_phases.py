"""Single phases of a whole-world dispatch, on the CPU: the host runtime built against the stand-in for HIP
(tests/host_stub) counts what each call launches.  A later phase goes on from the world's scratch only where that is its own
call's; after a dispatch that left no such state (the one launch) or another one's, the earlier phases run with it."""
import os

from tests.test_host_runtime_tsan import CSRC, build, run


def test_a_later_phase_runs_what_its_call_lacks(tmp_path):
    binary = build(str(tmp_path), os.path.join(CSRC, "ep_runtime.hip"), "phases_driver", sanitize=False,
                   driver="phases_driver.cpp")
    proc = run(binary)
    assert proc.returncode == 0, proc.stdout[-4000:]
    assert "ok (0 failed checks)" in proc.stdout
