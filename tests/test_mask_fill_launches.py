"""Mask sets' launches on the CPU emulation (AddressSanitizer): a fill whose
launch or event record fails keeps no state as if its mask had been written,
and one that copies no row makes one launch."""
import os
import subprocess

import emu_harness


def test_launches_and_failures_of_fills():
    exe = emu_harness.build("emu_fill")
    env = dict(os.environ)
    env.setdefault("ASAN_OPTIONS", "detect_leaks=0:abort_on_error=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stderr[-3000:]
