"""Where a step's workspaces live: the placement chosen at creation, its number
and what selects it again."""
from __future__ import annotations

import numpy as np
import pytest

from mjmlx_hip import capi, scenes
from test_gpu_compact import _states

pytestmark = pytest.mark.gpu

COMPACT = 7


# the batches of the rerun's bit comparisons, which start in small workspaces; 14
# boxes' full workspace does not fit LDS at all
@pytest.mark.parametrize("n,B,solver", [(8, 600, "CG"), (9, 513, "CG"), (11, 300, "CG"), (7, 800, "Newton"), (14, 257, "CG")])
def test_small_workspaces_have_a_number(n, B, solver):
    model = capi.Model(scenes.boxes_xml(n, 100 + n, solver=solver, iterations=16))
    rng = np.random.default_rng(n)
    q = _states(model, n, B, rng.random(B) < 0.1, rng)
    sim = capi.BatchedSim(model, B)
    assert sim.variant() == COMPACT
    out = []
    for v in (None, 1, COMPACT):
        assert v is None or sim.set_variant(v)
        assert v is None or sim.variant() == v
        sim.set_state(q, np.zeros((B, 6 * n), np.float32))
        sim.set_qacc_warmstart(np.zeros((B, 6 * n), np.float32))
        sim.step(None, 2)
        out.append(sim.state())
    for o in out[1:]:
        assert np.array_equal(out[0][0], o[0]) and np.array_equal(out[0][1], o[1])
    # what the autotuner reports is what it left and what selects it again
    choice = sim.autotune(2)
    assert choice == sim.variant() and sim.set_variant(choice)


def test_refused_where_the_sim_has_none():
    """A batch whose full workspaces are resident at once, and a small model."""
    for model, B in ((capi.Model(scenes.boxes_xml(8, 108)), 64), (capi.Model(scenes.quadruped_xml()), 600)):
        sim = capi.BatchedSim(model, B)
        v = sim.variant()
        assert v != COMPACT and not sim.set_variant(COMPACT) and sim.variant() == v
