"""GPU: a long token of text bytes passes as soon as a walk comes to a string's
text (after an escape): it costs no step per byte.  The bits are held by
test_mask_fill_launches.py and test_gpu_mask_states.py."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def test_plain_tokens_cost_no_step_per_byte():
    """16 rows after a backslash, 4,000 tokens that begin with an escape's letter: 8 bytes long against 200 bytes
    long, at most twice the time (launches of 10 us, which the host's own time moves; stepped byte by byte the long
    ones took 68 us)."""
    import torch

    from tachyon_amd.constrain import DeviceVocab, HostVocab, JsonConstraint, json_mask, pack_states

    c = JsonConstraint()
    c.advance(b'{"a": "x\\')
    states = torch.from_numpy(pack_states([c] * 16)).cuda()
    n = 4000
    mask = torch.zeros(16, n // 32, dtype=torch.int32, device="cuda")

    def us(length):
        v = DeviceVocab(HostVocab.from_tokens([b"bfnrt/"[t % 6:t % 6 + 1] + b"x" * (length - 1) if t % 64 == 0 else b"n"
                                               for t in range(n)], []))
        times = []
        for _ in range(9):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            for _ in range(50):
                json_mask(v, states, 16, n, mask, n // 32)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 20.0)
        assert (mask.cpu().numpy().view(np.uint32) == 0xFFFFFFFF).all()
        return sorted(times)[4]

    us(8)
    short, long = us(8), us(200)
    print(f"8 bytes {short:.1f} us, 200 bytes {long:.1f} us", flush=True)
    assert long < 2.0 * short
