"""
The read-back of a call's inputs (range check of the atomic numbers, parameter
tensors on the device): the same results whatever holds the parameters, the
same errors as a check before the launches, refused during stream capture.
"""

import pytest
import torch

import tad_dftd4_amd as d4
from tad_dftd4_amd import runtime, synth

pytestmark = pytest.mark.gpu

PARAM = {"s6": 1.0, "s8": 1.25, "s9": 1.0, "a1": 0.5, "a2": 5.0}


def _mol():
    numbers, positions, charge = synth.pack(synth.batch(5, 3, 5, 30))
    return numbers.cuda(), positions.cuda(), charge.cuda()


@pytest.mark.parametrize("dtype", [torch.float64, torch.float32, torch.float16])
@pytest.mark.parametrize("device", ["cpu", "cuda"])
def test_parameter_tensors(dtype, device):
    numbers, positions, charge = _mol()
    ref = d4.dftd4(numbers, positions, charge, PARAM)
    par = {k: torch.tensor(v, dtype=dtype, device=device) for k, v in PARAM.items()}
    par["a2"] = par["a2"].reshape(1)
    cut = d4.Cutoff(device=torch.device(device), dtype=dtype)
    # (the values are exact in 16 bits)
    assert torch.equal(ref, d4.dftd4(numbers, positions, charge, par, cutoff=cut))
    # a charge on the device, on the host and as a number are the same charge
    e = [d4.dftd4(numbers[0], positions[0], c, PARAM)
         for c in (charge[0], charge[0].cpu(), float(charge[0]))]
    assert torch.equal(e[0], e[1]) and torch.equal(e[0], e[2])


@pytest.mark.parametrize("bad", [-1, 104, 2**40])
@pytest.mark.parametrize("where", [0, 31, 2000])
def test_bad_numbers(bad, where):
    n = where + 1
    numbers = torch.ones(n, dtype=torch.int64, device="cuda")
    positions = torch.arange(3.0 * n, dtype=torch.float64, device="cuda").reshape(n, 3)
    numbers[where] = bad
    dev = {k: torch.tensor(v, device="cuda") for k, v in PARAM.items()}
    for call in (lambda: d4.dftd4(numbers, positions, 0.0, PARAM),
                 lambda: d4.dftd4(numbers, positions, 0.0, dev),
                 lambda: d4.dftd4(numbers, positions, 0.0, {"a1": 0.4}),
                 lambda: d4.dftd4_energy_gradient(numbers, positions, 0.0, PARAM),
                 lambda: d4.get_properties(numbers, positions),
                 lambda: d4.cn_d4(numbers, positions),
                 lambda: d4.D4Model(numbers).weight_references(torch.ones(n, device="cuda"))):
        with pytest.raises(ValueError, match="atomic numbers"):
            call()


def test_refused_in_capture():
    numbers, positions, charge = _mol()
    check = runtime.InputCheck(numbers)
    check.wait()
    check.wait()  # a second wait has nothing to wait for
    side = torch.cuda.Stream()
    with torch.cuda.stream(side):
        graph = torch.cuda.CUDAGraph()
        with pytest.raises(RuntimeError, match="captured"):
            with torch.cuda.graph(graph, stream=side):
                runtime.InputCheck(numbers)
    torch.cuda.synchronize()
    assert runtime.InputCheck(numbers).wait() == []
