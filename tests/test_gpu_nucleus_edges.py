"""Rows without top-k whose re-read passes meet their limits: rows that start
and end inside a 16-byte block, lengths around a tile and a bitmap stretch,
histories inside and past the table of penalized ids, masks, against the
oracle bit for bit (token, kept count, probability).  On the GPU, and the
short rows on the CPU emulation of the same sources."""
import numpy as np
import pytest

from tachyon_amd import workloads as wl

# usable ids, row stride, history length, masked
CASES = [(1027, 1029, 16, False), (1030, 1031, 0, True), (2051, 2053, 2100, False), (4098, 4099, 40, True)]
GPU_CASES = [(16387, 16389, 64, False), (32766, 32767, 2048, True), (33001, 33003, 2049, False),
             (151669, 151937, 300, False), (65539, 65541, 5000, True)]


def nucleus_case(usable, stride, history, masked, rows=7):
    rng = np.random.default_rng(usable + history)
    x = (rng.standard_normal((rows, stride)) * 1.5).astype(np.float32)
    p = wl.make_params(rows, temperature=1.1, top_p=0.97)
    p["top_p"][::3] = 1.0
    p["min_p"][4:5] = 1e-4
    ids = offs = mask = None
    if history:
        ids, offs = wl.uniform_histories(rng, rows, history, usable)
        ids[:8] = [0, 1, 2, 3, usable - 1, usable - 2, usable - 3, 0]  # the row's ends
        p["repetition_penalty"] = 1.2
        p["presence_penalty"][1::2] = -0.3
    if masked:
        mask = wl.pack_mask(rng.random((rows, usable)) < 0.6)
        p["flags"][::2] = wl.ROW_CONSTRAINED
    return wl.Workload(f"nucleus{usable}", x, usable, p, ids, offs, mask, wl.uniforms(rng, rows))


def agree(w, got):
    from oracle import pyoracle
    from parity import check

    check(w, got, pyoracle.sample_batch(w, nthreads=4), w.name)


@pytest.mark.gpu
@pytest.mark.parametrize("usable,stride,history,masked", CASES + GPU_CASES)
def test_nucleus_edges_on_the_gpu(usable, stride, history, masked):
    from tachyon_amd.device import SamplerContext, run_workload

    w = nucleus_case(usable, stride, history, masked)
    ctx = SamplerContext(max_rows=w.rows, max_vocab=usable)
    try:
        got = run_workload(ctx, w)
        assert ctx.status() == 0
    finally:
        ctx.close()
    agree(w, got)


@pytest.mark.parametrize("usable,stride,history,masked", CASES)
def test_nucleus_edges_on_the_cpu_emulation(usable, stride, history, masked):
    import emu_harness

    emu_harness.build()
    w = nucleus_case(usable, stride, history, masked, rows=3)
    agree(w, emu_harness.emu_sample(w))
