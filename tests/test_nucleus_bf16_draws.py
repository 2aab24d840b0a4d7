"""Rows of bf16-rounded logits (a value bin holds candidates of one value, all
rounding the same way) with draws that end deep in the tail: bit for bit
against the oracle, on the CPU emulation of the kernels and on the GPU, and
within a small multiple of the time of continuous logits."""
import numpy as np
import pytest

from tachyon_amd import workloads as wl


def bf16_rows(rows, usable, sigma, top_p, seed=23):
    rng = np.random.default_rng(seed)
    x = rng.standard_normal((rows, usable), dtype=np.float32) * np.float32(sigma)
    x = ((x.view(np.uint32) + 0x8000) & np.uint32(0xFFFF0000)).view(np.float32)
    p = wl.make_params(rows, temperature=1.0, top_p=top_p)
    u = np.linspace(0.99, 0.999999, rows).astype(np.float32)
    return wl.Workload(f"bf16_{usable}", x, usable, p, None, None, None, u)


def agree(w, got):
    from oracle import pyoracle
    from parity import check

    check(w, got, pyoracle.sample_batch(w, nthreads=4), w.name)


@pytest.mark.parametrize("sigma,top_p", [(2.0, 1.0), (1.0, 0.98)])
def test_bf16_draws_on_the_cpu_emulation(sigma, top_p):
    import emu_harness

    emu_harness.build()
    w = bf16_rows(4, 20000, sigma, top_p)
    agree(w, emu_harness.emu_sample(w))


@pytest.mark.gpu
@pytest.mark.parametrize("sigma,top_p", [(1.0, 1.0), (2.0, 1.0), (2.0, 0.98), (3.0, 1.0)])
def test_bf16_draws_on_the_gpu(sigma, top_p):
    import torch

    from tachyon_amd.device import SamplerContext, run_workload

    torch.cuda.init()  # before the library's first call
    w = bf16_rows(12, 151936, sigma, top_p)
    ctx = SamplerContext(max_rows=w.rows, max_vocab=w.usable)
    try:
        got = run_workload(ctx, w)
        assert ctx.status() == 0
    finally:
        ctx.close()
    agree(w, got)


@pytest.mark.gpu
@pytest.mark.parametrize("sigma,top_p", [(2.0, 0.98), (3.0, 1.0)])
def test_bf16_draws_cost_no_round_a_bin(sigma, top_p):
    """256 rows, one a CU, so the worst row's time: at most twice that of the same rows before rounding.  (Where the
    draw's estimate was off, every bin up to a crossing's real place asked for a pass of its own: four to five times.)"""
    import torch

    from tachyon_amd.device import DeviceBatch, Outputs, SamplerContext

    rows, usable = 256, 151936
    gen = torch.Generator(device="cuda").manual_seed(23)
    x = torch.randn(rows, usable, generator=gen, device="cuda") * sigma
    p = wl.make_params(rows, temperature=1.0, top_p=top_p)
    ctx = SamplerContext(rows, usable)
    out = Outputs(rows, 1)

    def ms(logits):
        b = DeviceBatch(logits=logits, usable=usable, params=torch.from_numpy(p.view(np.uint8)).cuda(), hist_ids=None,
                        hist_offsets=None, mask=None, uniforms=torch.linspace(0.99, 0.999999, rows, device="cuda"),
                        top_stride=1, row_kinds=0, dist_kinds=0)
        times = []
        for _ in range(4):
            s, e = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            s.record()
            ctx.sample(b, out, with_logprobs=False)
            e.record()
            e.synchronize()
            times.append(s.elapsed_time(e))
        return min(times)

    try:
        plain, rounded = ms(x), ms(x.bfloat16().float())
    finally:
        ctx.close()
    print(f"sigma {sigma} top_p {top_p}: {plain:.2f} ms, rounded to bf16 {rounded:.2f} ms", flush=True)
    assert rounded < 2.0 * plain
