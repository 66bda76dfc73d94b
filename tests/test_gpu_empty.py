"""
Molecules without atoms (all padding) inside a batch: zero energy, gradient and
charges, and the other molecules as in a batch of their own, bit for bit. The
padded lengths take the one-pass three-body kernel, the paired charge solve and
the screened kernel with the tiled solve. Parameter gradients are sums over the
batch whose grouping depends on its size: at most some 1e3 partials, so 1e-12
of the largest is far above the rounding of another order.
"""

import pytest
import torch

from tad_dftd4_amd import runtime, synth

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("d4s", [False, True])
@pytest.mark.parametrize("pad", [24, 64, 200, 300])
def test_empty_molecules(pad, d4s):
    print(f"[case] empty molecules, padded to {pad}, d4s={d4s}", flush=True)
    mols = synth.batch(11, 4, max(2, pad // 2), pad)
    numbers, positions, charge = (t.cuda() for t in synth.pack(mols, pad_to=pad))
    at = torch.tensor([1, 2, 4, 6], device="cuda")  # 0, 3, 5 and 7 are empty
    n8 = torch.zeros(8, pad, dtype=torch.int64, device="cuda")
    x8 = torch.zeros(8, pad, 3, dtype=torch.float64, device="cuda")
    q8 = torch.zeros(8, dtype=torch.float64, device="cuda")
    n8[at], x8[at], q8[at] = numbers, positions, charge
    empty = torch.ones(8, dtype=torch.bool, device="cuda")
    empty[at] = False
    kp = runtime.KernelParams(s8=1.2, a1=0.4, a2=5.0, cutoff_disp3=25.0, d4s=d4s)

    e, g, _ = runtime.energy_gradient(numbers, positions, charge, kp)
    e8, g8, _ = runtime.energy_gradient(n8, x8, q8, kp)
    assert torch.equal(e8[at], e) and torch.equal(g8[at], g)
    assert not e8[empty].any() and not g8[empty].any()

    f, ws = runtime.forward(numbers, positions, charge, kp)
    f8, ws8 = runtime.forward(n8, x8, q8, kp)
    assert torch.equal(f8[at], f) and not f8[empty].any()
    gb, gp = runtime.backward(numbers, positions, charge, kp, ws, params=True)
    gb8, gp8 = runtime.backward(n8, x8, q8, kp, ws8, params=True)
    assert torch.equal(gb8[at], gb) and not gb8[empty].any()
    assert (gp8 - gp).abs().max().item() <= 1e-12 * gp.abs().max().item()

    if not d4s:
        for a, a8 in zip(runtime.properties(numbers, positions, charge, kp),
                         runtime.properties(n8, x8, q8, kp)):
            assert torch.equal(a8[at], a) and not a8[empty].any()
