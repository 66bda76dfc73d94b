"""
The shipped launch-shape table against the kernels it is for: the 8 x 8 pair
tiles of the one-pass three-body kernel beat the 16 x 16 ones at every length
and in both modes (energies of 640 molecules of 97-192 atoms 1.20 against 1.53
ms, of 480 of 129-256 atoms 2.50 against 2.94), so an entry that names 16 x 16
was measured on other kernels and makes its callers slower.
"""

from pathlib import Path

import pytest

from tad_dftd4_amd import tune


@pytest.mark.parametrize("mode", tune.MODES)
def test_no_slower_tile(mode):
    table = tune.ShapeTable.load(Path(tune.__file__).with_name("shapes_gfx950.json"))
    assert all(tile in (0, 8) for _, _, tile in table.entries[mode])
    for n_max, times in table.timings[mode].items():
        if int(n_max) <= tune.ONE_PASS_MAX:
            eight = min(v for k, v in times.items() if k.endswith("x8"))
            assert eight < min(v for k, v in times.items() if k.endswith("x16"))
