"""
EEQ charges and their adjoint over the sizes where the solve changes shape:
edges of the 16-column blocks, of the 64-entry pieces of the substitutions, of
the wave count and of the LDS placement, with and without padding atoms.

Charges against the oracle's dense solve. Both sides round an n x n system in
64 bits: the error is at most about n eps cond |q|, with n <= 201 and condition
numbers below 1e4 (diagonal 0.5-2, off-diagonal < 0.4) about 4e-10 in the
worst case and some 1e-13 typically; 1e-10 here. Gradients (through the
adjoint) against the same call with the pivoted-LU solve, whose other kernels
are identical: 1e-11 Eh/bohr on gradients of 1e-3.
"""

import numpy as np
import pytest
import torch

from oracle import dense
from tad_dftd4_amd import runtime, synth

pytestmark = pytest.mark.gpu

SIZES = (1, 2, 15, 16, 17, 33, 63, 64, 65, 112, 128, 129, 140, 141, 191, 196, 197, 200, 201)


def _batch(n, pad):
    rng = np.random.default_rng(100 + n)
    mols = [synth.molecule(rng, k, synth.MIX_HCNO, 2.8, (-1, 0, 1)) for k in {n, max(1, n - 9)}]
    mols.append(mols[0])
    numbers, positions, charge = synth.pack(mols, pad_to=pad)
    if n > 4:
        numbers[-1, n // 2] = 0  # an inner padding atom
    return numbers, positions, charge


@pytest.mark.parametrize("n", SIZES)
def test_charges_and_adjoint(n):
    print(f"[case] EEQ n = {n}", flush=True)
    for pad in {n, 201}:
        numbers, positions, charge = _batch(n, pad)
        ref = dense.eeq_charges(numbers, positions, charge)
        dev = [t.cuda() for t in (numbers, positions, charge)]
        q = runtime.properties(*dev, runtime.KernelParams())[1].cpu()
        assert (q - ref).abs().max().item() < 1e-10
        e, g, ws = runtime.energy_gradient(*dev, runtime.KernelParams())
        assert not runtime.molecule_status(ws, len(numbers)).any()
        e_lu, g_lu, _ = runtime.energy_gradient(*dev, runtime.KernelParams(force_lu=True))
        assert (e - e_lu).abs().max().item() < 1e-13
        assert (g - g_lu).abs().max().item() < 1e-11


def test_batches_in_and_out_of_order():
    # more molecules than one per CU are solved by size, fewer in batch order,
    # with the same bits
    rng = np.random.default_rng(7)
    mols = [synth.molecule(rng, int(k), synth.MIX_HCNO, 2.8, (0, 1))
            for k in rng.integers(2, 40, size=300)]
    numbers, positions, charge = (t.cuda() for t in synth.pack(mols))
    kp = runtime.KernelParams()
    e, g, _ = runtime.energy_gradient(numbers, positions, charge, kp)
    for part in (slice(0, 100), slice(100, 300)):
        ep, gp, _ = runtime.energy_gradient(numbers[part].contiguous(),
                                            positions[part].contiguous(),
                                            charge[part].contiguous(), kp)
        assert torch.equal(e[part], ep) and torch.equal(g[part], gp)


TILED = (1, 15, 16, 62, 63, 64, 65, 80, 126, 127, 128, 129, 255, 256, 257, 320, 511, 513)


@pytest.mark.parametrize("n", TILED)
def test_tiled_charges_and_adjoint(n):
    # edges of the 64-column blocks (the border rows fall into the last diagonal
    # tile for 64 k + 1 .. 64 k + 62 atoms, across it for 63, behind it for 64)
    # and of the 256-entry substitutions; same bounds as above, n = 513
    print(f"[case] tiled EEQ n = {n}", flush=True)
    for pad in {n, n + 3}:
        numbers, positions, charge = _batch(n, pad)
        ref = dense.eeq_charges(numbers, positions, charge)
        dev = [t.cuda() for t in (numbers, positions, charge)]
        kp = runtime.KernelParams(force_tiled=True)
        q = runtime.properties(*dev, kp)[1].cpu()
        assert (q - ref).abs().max().item() < 1e-10
        e, g, ws = runtime.energy_gradient(*dev, kp)
        assert not runtime.molecule_status(ws, len(numbers)).any()
        e_lu, g_lu, _ = runtime.energy_gradient(
            *dev, runtime.KernelParams(force_tiled=True, force_lu=True))
        assert (e - e_lu).abs().max().item() < 1e-13
        assert (g - g_lu).abs().max().item() < 1e-11
