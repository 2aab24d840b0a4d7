"""GPU: tsm_json_mask where its workgroups meet their limits: batches of one
row, of one more than a workgroup's states and of several groups, rows in the
same and in different states (also ones that only rejected bytes leave), and
tokens whose block exceeds the workgroup's stage, bit for bit against the host
automaton (tsm_json_accepts, itself held to the oracle by test_mask_cpu.py)."""
import numpy as np
import pytest

from tachyon_amd import workloads as wl

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rows,long_tokens", [(1, False), (255, True), (257, False), (700, True)])
def test_masks_at_the_workgroups_limits(rows, long_tokens):
    import torch

    from tachyon_amd.constrain import DeviceVocab, HostVocab, JsonConstraint, json_mask, pack_states

    rng = np.random.default_rng(rows)
    toks, special = wl.json_vocab(700, seed=11)
    if long_tokens:  # tokens 300..511: over 16 KB in one block of 256
        for i in range(300, 512):
            toks[i] = b'"' + b"x" * 96 + (b'"' if i % 2 else b"")
    hv = HostVocab.from_tokens(toks, special)
    states = []
    for p in wl.json_prefixes(min(rows, 300), seed=rows):
        c = JsonConstraint()
        c.advance(p)
        if rng.random() < 0.1:
            c.advance(rng.integers(0, 256, 5).astype(np.uint8).tobytes())
        states.append(c)
    while len(states) < rows:
        states.append(states[int(rng.integers(0, len(states)))])
    usable = 690
    nw = (usable + 31) // 32
    mask = torch.full((rows, nw + 1), 0x5A5A5A5A, dtype=torch.int32, device="cuda")
    json_mask(DeviceVocab(hv), torch.from_numpy(pack_states(states)).cuda(), rows, usable, mask, nw + 1)
    got = mask.cpu().numpy().view(np.uint32)
    known = {}
    for r, c in enumerate(states):
        key = c.packed()
        if key not in known:
            ok = np.array([[not hv.is_special(t) and len(toks[t]) > 0 and c.accepts(toks[t]) for t in range(usable)]])
            known[key] = wl.pack_mask(ok)[0]
        assert (got[r, :nw] == known[key]).all(), (rows, r)
        assert got[r, nw] == 0x5A5A5A5A
