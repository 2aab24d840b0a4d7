"""The mask producer's automaton table and its kernel on the CPU emulation
(AddressSanitizer): the table against the byte-by-byte automaton, and whole
masks for batches past one workgroup's states and tokens past its stage."""
import os
import subprocess

import emu_harness


def test_table_and_kernel_on_the_cpu_emulation():
    exe = emu_harness.build("emu_json")
    env = dict(os.environ)
    env.setdefault("ASAN_OPTIONS", "detect_leaks=0:abort_on_error=1")
    r = subprocess.run([exe], capture_output=True, text=True, timeout=600, env=env)
    assert r.returncode == 0 and r.stdout.strip() == "ok", r.stderr[-3000:]
