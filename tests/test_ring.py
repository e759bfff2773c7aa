"""The command ring between a processor's callers and its ring thread, alone on
the CPU, plain and under ThreadSanitizer: two producers with a thread that
drains, a full ring whose producers go to sleep, wrap-around in the middle of a
command, an end with commands left, and pauses around the polling times; and that
every failed submission is reported by the flush it belongs to, and timed waits
end at their timeout.  A lost
wake-up hangs the probe and fails by its time limit."""
import os
import subprocess

import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


@pytest.fixture(scope="module", params=["plain", "thread"])
def probe(request, tmp_path_factory):
    out = str(tmp_path_factory.mktemp("ring") / request.param)
    flags = ["-O2"] if request.param == "plain" else ["-O1", "-g", "-fsanitize=thread"]
    subprocess.run(["g++", "-std=c++17", "-pthread", *flags, "-o", out, os.path.join(ROOT, "tests", "ring_probe.cpp")],
                   check=True)
    if request.param == "thread":
        # Some kernels place memory where ThreadSanitizer's own mappings must lie.
        run = subprocess.run([out, "0", "1"], capture_output=True, text=True, timeout=100)
        if "unexpected memory mapping" in run.stderr:
            pytest.skip("ThreadSanitizer does not start on this kernel: " + run.stderr[:200])
    return out


@pytest.mark.parametrize("mode,count", [(0, 20000), (1, 12000), (2, 6000), (3, 200), (2, 1), (0, 1), (4, 0), (5, 0)])
def test_ring(probe, mode, count):
    run = subprocess.run([probe, str(mode), str(count)], capture_output=True, text=True, timeout=100)
    assert run.returncode == 0 and run.stdout.strip() == "ok", run.stdout + run.stderr[-3000:]
