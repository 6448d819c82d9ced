"""The threads of the host transfers, on the CPU: transfer.hpp itself with the
runtime's calls replaced (tests/transfer_threads.cpp).

A transfer must not wait for a helper thread that has not got a processor yet:
right after an OpenMP region, whose workers spin on every one, that took
milliseconds.  Held back for good, every helper leaves the whole transfer to the
calling thread, and comes too late to touch it.  Values and ghost layers are
right with and without helpers, and ThreadSanitizer finds nothing.
"""
import shutil
import subprocess
from pathlib import Path

import pytest

ROOT = Path(__file__).resolve().parents[1]
HIPCC = shutil.which("hipcc") or "/opt/rocm/bin/hipcc"

pytestmark = pytest.mark.skipif(not Path(HIPCC).exists(), reason="hipcc not found")


def _run(tmp_path, mode, rounds, *flags):
    exe = tmp_path / "transfer_threads"
    cmd = [HIPCC, "-std=c++17", "-O1", "--offload-arch=gfx950", "-DHOWMHD_EXACT=1", f"-I{ROOT / 'include'}",
           f"-I{ROOT / 'how-mhd-kokkos_amd' / 'csrc'}", *flags, str(ROOT / "tests" / "transfer_threads.cpp"), "-rdynamic",
           "-ldl", "-o", str(exe)]
    build = subprocess.run(cmd, capture_output=True, text=True, timeout=300)
    if build.returncode != 0 and flags:
        pytest.skip("sanitizer runtime not available: " + build.stderr[-300:])
    assert build.returncode == 0, build.stderr[-3000:]
    r = subprocess.run([str(exe), mode, str(rounds)], capture_output=True, text=True, timeout=60)
    if "FATAL: ThreadSanitizer" in r.stderr:  # (a memory layout it does not know)
        pytest.skip(r.stderr[-300:])
    assert r.returncode == 0 and "WRONG" not in r.stdout, r.stdout[-2000:] + r.stderr[-3000:]


@pytest.mark.parametrize("mode,rounds", [("held", 1), ("free", 4)])
def test_late_helpers(mode, rounds, tmp_path):
    _run(tmp_path, mode, rounds)


def test_helpers_under_thread_sanitizer(tmp_path):
    _run(tmp_path, "free", 1, "-Xarch_host", "-fsanitize=thread", "-g")
