"""
Coordination numbers and chain pass by block rows (few molecules) against the
pass by molecules (many): the same pair terms summed in the same order, so the
bits are the same. The batch holds more molecules than its padded length, the
single call one, with padding at the end and inside.
"""

import numpy as np
import pytest
import torch

from tad_dftd4_amd import runtime, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d4s", [False, True])
@pytest.mark.parametrize("n", [2, 7, 8, 9, 17, 63, 64, 65, 130, 255])
def test_block_rows_and_molecules_same_bits(n, d4s):
    print(f"[case] block rows n = {n}, d4s {d4s}", flush=True)
    rng = np.random.default_rng(600 + n)
    N = n + 1 if n != 64 else 64
    mols = [synth.molecule(rng, k, synth.MIX_HCNO, 2.8, (-1, 0, 1)) for k in [n] + [2] * N]
    numbers, positions, charge = synth.pack(mols, pad_to=N)
    if n > 8:
        numbers[0, n // 2] = 0
    many = [t.cuda() for t in (numbers, positions, charge)]
    one = [t[:1].contiguous() for t in many]
    assert len(mols) > N  # by molecules; one molecule goes by block rows
    kp = runtime.KernelParams(s8=1.2, a1=0.4, a2=5.0, d4s=d4s)
    if not d4s:  # (the property call evaluates the D4 model)
        for a, b in zip(runtime.properties(*many, kp)[:2], runtime.properties(*one, kp)[:2]):
            assert torch.equal(a[:1], b)
    e, g, _ = runtime.energy_gradient(*many, kp)
    e1, g1, _ = runtime.energy_gradient(*one, kp)
    assert torch.equal(e[:1], e1) and torch.equal(g[:1], g1)
    q = 0.1 * torch.randn(e.shape, dtype=torch.float64, device="cuda")
    ef, ws = runtime.forward(*many, kp, q=q)
    gb = runtime.backward(*many, kp, ws, q=q)
    q1 = q[:1].contiguous()
    ef1, ws1 = runtime.forward(*one, kp, q=q1)
    gb1 = runtime.backward(*one, kp, ws1, q=q1)
    assert torch.equal(ef[:1], ef1) and torch.equal(gb[:1], gb1)
