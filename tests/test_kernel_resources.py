"""Occupancy of g2p in 3D: five waves per SIMD in both particle layouts (96
registers, of 512 for the waves of a SIMD, given out eight at a time), and
nothing spilled there and at the six waves that the tuning can ask for."""
import pytest

from tests.kernel_resources import kernel_resources


@pytest.mark.parametrize("packed", ["false", "true"])
@pytest.mark.parametrize("waves,registers", [(1, 96), (6, 80)])
def test_g2p_occupancy(packed, waves, registers):
    res = kernel_resources()
    k = res[f"k_g2p<3, {packed}, {waves}, false>"]
    assert k["spills"] == 0
    assert k["vgprs"] <= registers
    # the grid operator inside: not offered at six waves, where it would spill
    assert f"k_g2p<3, {packed}, 6, true>" not in res
    assert res[f"k_g2p<3, {packed}, 1, true>"]["spills"] == 0
