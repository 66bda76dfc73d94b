"""
D4S weights by element: the pair passes take both atoms' Gaussian weights from
per-element tables (contraction vectors of the partner, LDS rows of the atom)
where a molecule has at most 32 distinct elements, and form them per pair
otherwise. Both against the oracle in one batch, at one, two and four rows per
wave, energies, fused and weighted gradients.

Tolerances as for the other oracle comparisons: 1e-10 Eh, 1e-9 Eh/bohr.
"""

import numpy as np
import pytest
import torch

from oracle import dense
from tad_dftd4_amd import runtime, synth

pytestmark = pytest.mark.gpu

PARAM = {"s6": 1.0, "s8": 1.2, "s9": 1.0, "a1": 0.40, "a2": 5.0}
CUT = {"disp2": 50.0, "disp3": 25.0, "cn_eeq": 25.0}


@pytest.mark.parametrize("row_lanes", [16, 32, 64])
def test_element_tables_and_pairs(row_lanes):
    print(f"[case] D4S element tables, {row_lanes} lanes per row", flush=True)
    rng = np.random.default_rng(810)
    mols = []
    for n, elements in ((44, 33), (40, 32), (23, 17), (5, 1)):
        mol = synth.molecule(rng, n, synth.MIX_Z54, 3.0, (0,))
        numbers = np.array([1 + k % elements for k in range(n)])  # Z = 1 .. elements
        mols.append(synth.Molecule(numbers, mol.positions, 0))
    numbers, positions, charge = synth.pack(mols, pad_to=47)
    dev = [t.cuda() for t in (numbers, positions, charge)]
    kp = runtime.KernelParams(**PARAM, cutoff_disp2=50.0, cutoff_disp3=25.0, cutoff_eeq=25.0,
                              d4s=True, row_lanes=row_lanes)
    e, g, _ = runtime.energy_gradient(*dev, kp)
    ef, ws = runtime.forward(*dev, kp)
    w = torch.linspace(0.5, 1.5, 47, dtype=torch.float64).expand(4, 47).contiguous()
    gb = runtime.backward(*dev, kp, ws, w.cuda())
    par = {k: torch.tensor(v, dtype=torch.float64) for k, v in PARAM.items()}
    for k, mol in enumerate(mols):
        n = len(mol.numbers)
        pos = torch.tensor(mol.positions).requires_grad_(True)
        eo = dense.dftd4(torch.tensor(mol.numbers), pos, 0.0, par, cutoff=CUT, model="d4s")
        (go,) = torch.autograd.grad(eo.sum(), pos, retain_graph=True)
        (gw,) = torch.autograd.grad((eo * w[k, :n]).sum(), pos)
        for x in (e, ef):
            assert (x[k, :n].cpu() - eo.detach()).abs().max().item() < 1e-10
        assert (g[k, :n].cpu() - go).abs().max().item() < 1e-9
        assert (gb[k, :n].cpu() - gw).abs().max().item() < 1e-9
