"""The staged host copies (pmp_copy.hip) on the CPU: tests/native/copy_selftest.cpp
drives them against a simulated HIP runtime whose streams run behind their
callers, built with AddressSanitizer + UndefinedBehaviorSanitizer and with
ThreadSanitizer.  No GPU."""
import os
import subprocess

import pytest

NATIVE = os.path.join(os.path.dirname(os.path.abspath(__file__)), "native")
ENV = dict(os.environ, ASAN_OPTIONS="detect_leaks=1", UBSAN_OPTIONS="halt_on_error=1:print_stacktrace=1",
           TSAN_OPTIONS="halt_on_error=1")


@pytest.mark.parametrize("san", ["asan", "tsan"])
@pytest.mark.parametrize("part", ["pitched", "until", "shared", "streams", "maps", "together"])
def test_copies(san, part):
    r = subprocess.run(["make", "-s", "-C", NATIVE, f"build/copy_selftest_{san}"], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([os.path.join(NATIVE, "build", f"copy_selftest_{san}"), part], capture_output=True, text=True,
                       timeout=100, env=ENV)
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer cannot map its shadow memory on this kernel")
    assert r.returncode == 0 and f"{part} ok" in r.stdout, f"rc {r.returncode}\n{r.stdout}\n{r.stderr[-6000:]}"


def test_scheduler_under_tsan():
    """The serving scheduler's own self-test under ThreadSanitizer (tests/native/host_selftest.cpp)."""
    r = subprocess.run(["make", "-s", "-C", NATIVE, "build/host_selftest_tsan"], capture_output=True, text=True,
                       timeout=300)
    assert r.returncode == 0, r.stderr[-3000:]
    r = subprocess.run([os.path.join(NATIVE, "build", "host_selftest_tsan")], capture_output=True, text=True,
                       timeout=120, env=ENV)
    if "unexpected memory mapping" in r.stderr:
        pytest.skip("ThreadSanitizer cannot map its shadow memory on this kernel")
    assert r.returncode == 0 and "host_selftest: ok" in r.stdout, f"rc {r.returncode}\n{r.stdout}\n{r.stderr[-6000:]}"
