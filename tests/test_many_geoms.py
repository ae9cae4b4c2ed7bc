"""More geoms than 16 bits number: the pair records hold both indices whole."""
from __future__ import annotations

import numpy as np

import emu


def test_pair_of_geoms_beyond_65535():
    """A ball whose geom comes after 66000 others, which touch nothing, lands on
    the floor like one alone (the model compiles in about 15 s: all pairs are
    looked at)."""
    def drop(n):
        sim = emu.EmuSim('<mujoco><worldbody><geom type="plane" size="5 5 0.1"/><body pos="0 0 0.09"><freejoint/>'
                         + '<geom size="0.01" mass="0" contype="0" conaffinity="0"/>' * n
                         + '<geom size="0.1" mass="1"/></body></worldbody></mujoco>', 1)
        sim.step(None, 4)
        return (*sim.get_state(), sim.stats()["ncon"], sim.stats()["niter"])

    one, many = drop(0), drop(66000)
    assert one[3][0] == 1
    for a, b in zip(one, many):
        assert np.array_equal(a, b)
