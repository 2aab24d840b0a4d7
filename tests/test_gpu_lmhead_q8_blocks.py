"""GPU: the Q8 lm_head's 32-value block kernel (batches of more than 32 rows)
where it can go wrong, bit for bit against the oracle: rows around its tiles,
block counts that are not whole chunks, scales that are not 8-byte aligned, and
logits that are zero (rows of zeros, weights of zeros, scales of either sign),
whose sign only the exact recomputation gives."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows", [33, 64, 65, 129, 257])
@pytest.mark.parametrize("dim,shift", [(32, 0), (96, 0), (160, 1), (256, 0), (1024, 2), (1056, 0)])
def test_q8_blocks_bit_exact(rows, dim, shift):
    import torch

    from oracle import pyoracle
    from tachyon_amd.lmhead import lm_head_q8

    vocab = 301
    rng = np.random.default_rng(rows * 10000 + dim)
    x = (rng.standard_normal((rows, dim)) * 2.0).astype(np.float32)
    x[::7] = 0.0                                   # zero rows
    x[1::11, : dim // 2] = 0.0
    g = (1.0 + 0.2 * rng.standard_normal(dim)).astype(np.float32)
    wq = rng.integers(-128, 128, (vocab, dim)).astype(np.int8)
    ws = (0.002 * rng.standard_normal((vocab, dim // 32))).astype(np.float16)
    ws[::5] = -np.abs(ws[::5])                     # ids whose every scale is negative
    wq[::6] = 0                                    # ids without weights
    wq[3::8, : dim // 2] = 0
    ws[4::9] = np.float16(-0.0)
    bits = ws.view(np.uint16)
    buf = torch.zeros(bits.size + 8, dtype=torch.int16, device="cuda")
    wsc = buf[shift:shift + bits.size].view(vocab, dim // 32)  # 2 * shift bytes off an aligned address
    wsc.copy_(torch.from_numpy(bits.view(np.int16)))
    out = torch.full((rows, vocab + 3), 7.0, dtype=torch.float32, device="cuda")
    lm_head_q8(torch.from_numpy(x).cuda(), torch.from_numpy(g).cuda(), 1e-6, torch.from_numpy(wq).cuda(), wsc, out=out)
    got = out.cpu().numpy()
    want = pyoracle.lm_head_q8(x, g, 1e-6, wq, bits)
    assert np.array_equal(got[:, :vocab].view(np.uint32), want.view(np.uint32))
    assert (got[:, vocab:] == 7.0).all()
