"""GPU: the Q8 lm_head's zero logits in batches of more than 32 rows, whose sign
the 32-value block kernel settles apart from its sums: rows and ids of zeros
under scales of every kind, rows whose scales let products underflow, sums that
cancel, bit for bit against the oracle; and padding costs no multiple of the
call's time."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def scales(rng, vocab, nb):
    """A kind of scales per id: any sign, all negative, all -0, all +0, all positive, negative but one +0 or one
    positive."""
    ws = (0.002 * rng.standard_normal((vocab, nb))).astype(np.float16)
    kind = np.arange(vocab) % 7
    ws[kind == 1] = -np.abs(ws[kind == 1])
    ws[kind == 2] = np.float16(-0.0)
    ws[kind == 3] = np.float16(0.0)
    ws[kind == 4] = np.abs(ws[kind == 4])
    ws[kind >= 5] = -np.abs(ws[kind >= 5])
    ws[kind == 5, nb // 2] = np.float16(0.0)
    ws[kind == 6, nb - 1] = np.float16(2.0 ** -24)
    return ws


def call(x, g, wq, bits, out):
    import torch

    from tachyon_amd.lmhead import lm_head_q8

    return lm_head_q8(x, g, 1e-6, torch.from_numpy(wq).cuda(), torch.from_numpy(bits.view(np.int16)).cuda(), out=out)


@pytest.mark.parametrize("rows,dim,vocab", [(33, 32, 131), (64, 160, 300), (65, 1056, 129), (128, 4096, 290),
                                            (130, 96, 515), (257, 1024, 260)])
def test_signs_of_zero_logits(rows, dim, vocab):
    import torch

    from oracle import pyoracle

    rng = np.random.default_rng(rows + dim)
    nb = dim // 32
    x = (rng.standard_normal((rows, dim)) * 2.0).astype(np.float32)
    x[::3] = 0.0                            # padding
    x[1::6] = np.sign(x[1::6])              # every block alike: products of opposite ids cancel
    g = np.ones(dim, np.float32)
    if nb > 1:
        g[32:64] = np.float32(1e-38)        # the rows' scales there are below any normal product
        x[2::9, 64:] = 0.0
        x[2::9, :32] = 0.0                  # rows with nothing but such a block
    wq = rng.integers(-128, 128, (vocab, dim)).astype(np.int8)
    wq[(np.arange(vocab) // 7) % 3 == 0] = 0   # ids without weights, under every kind of scales
    wq[1::11, : dim // 2] = 0
    wq[5::17] = np.where(np.arange(dim) % 2, 1, -1)
    bits = scales(rng, vocab, nb).view(np.uint16)
    out = torch.full((rows, vocab + 3), 7.0, dtype=torch.float32, device="cuda")
    call(torch.from_numpy(x).cuda(), torch.from_numpy(g).cuda(), wq, bits, out)
    got = out.cpu().numpy()
    want = pyoracle.lm_head_q8(x, g, 1e-6, wq, bits)
    zero = want == 0.0
    signs = np.signbit(want[zero])
    assert signs.any() and not signs.all()  # the oracle has both
    assert np.array_equal(got[:, :vocab].view(np.uint32), want.view(np.uint32))
    assert (got[:, vocab:] == 7.0).all()


@pytest.mark.parametrize("rows", [48, 128, 256])
def test_padding_costs_no_multiple_of_the_time(rows):
    """Zero rows, and zero ids under negative scales, against dense inputs: at most twice the time (a tile's notes
    are one look through its scales; computing each zero logit again took 30 to 300 times)."""
    import torch

    from tachyon_amd.lmhead import lm_head_q8

    dim, vocab = 4096, 32000
    gen = torch.Generator(device="cuda").manual_seed(rows)
    x = torch.randn(rows, dim, generator=gen, device="cuda")
    g = torch.ones(dim, device="cuda")
    w = torch.randint(-127, 128, (vocab, dim), generator=gen, device="cuda", dtype=torch.int8)
    ws = (0.001 * torch.randn(vocab, dim // 32, generator=gen, device="cuda")).half().view(torch.int16)
    out = torch.empty(rows, vocab, device="cuda")

    def us():
        times = []
        for _ in range(7):
            a, b = torch.cuda.Event(enable_timing=True), torch.cuda.Event(enable_timing=True)
            a.record()
            lm_head_q8(x, g, 1e-6, w, ws, out=out)
            b.record()
            b.synchronize()
            times.append(a.elapsed_time(b) * 1000.0)
        return sorted(times)[3]

    us()
    dense = us()
    x[rows // 2:] = 0.0
    padded = us()
    w[-267:] = 0
    ws[-267:] |= -32768
    ids = us()
    print(f"{rows} rows: dense {dense:.1f} us, half the rows zero {padded:.1f}, and 267 ids zero {ids:.1f}", flush=True)
    assert padded < 2.0 * dense and ids < 2.0 * dense
