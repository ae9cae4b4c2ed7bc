"""More bodies than lanes: the level-by-level stages go through the levels' lists.

Chains whose bodies are mostly welded (few dofs: such models run in the kernels
for any size from 65 bodies on), on 64 and on 32 lanes, and a hub of more
children than lanes, one level that takes two rounds. One step against the
oracle, to the parity tests' bar."""
from __future__ import annotations

import numpy as np
import pytest

import ref64
import states
from mjmlx_hip import capi

pytestmark = pytest.mark.gpu


def _link(pos, joint, inner=""):
    j = f'<joint type="hinge" axis="{joint}" damping="0.02" armature="0.001"/>' if joint else ""
    return (f'<body pos="{pos}">{j}<geom type="capsule" fromto="0 0 0 0 0 -0.1" size="0.02" density="500" '
            f'contype="0" conaffinity="0"/>{inner}</body>')


def _xml(bodies):
    return ('<mujoco><compiler angle="radian"/><option timestep="0.002" iterations="20"/><worldbody>' + bodies
            + "</worldbody></mujoco>")


def _chains(k, n, every):
    out = ""
    for c in range(k):
        inner = ""
        for i in reversed(range(n)):
            joint = ("1 0 0" if i % 2 else "0 1 0") if i % every == 0 else ""
            inner = _link(f"{0.3 * c} 0 3" if i == 0 else "0 0 -0.1", joint, inner)
        out += inner
    return _xml(out)


def _hub(n):
    leaves = "".join(_link(f"{0.05 * i:.2f} 0.1 0", "0 1 0" if i % 4 == 0 else "") for i in range(n))
    return _xml(_link("0 0 2", "1 0 0", leaves))


@pytest.mark.parametrize("name,bodies,variant", [("chains", 80, None), ("chains", 80, 1), ("hub", 71, None),
                                                 ("hub", 71, 2), ("half", 48, None), ("half", 48, 5)])
def test_one_step(name, bodies, variant):
    xml = {"chains": _chains(4, 20, 4), "hub": _hub(70), "half": _chains(2, 24, 6)}[name]
    model, B = capi.Model(xml), 6
    assert int(model.info.nbody) == bodies + 1 and model.nv <= 20
    sim = capi.BatchedSim(model, B)
    assert variant is None or sim.set_variant(variant)
    assert name != "half" or variant == 5 or sim.variant() not in (5, 6)  # more bodies than half a wave's lanes
    rng = np.random.default_rng(1)
    q, v = (rng.uniform(-0.3, 0.3, (B, model.nv)).astype(np.float32) for _ in range(2))
    sim.set_state(q, v)
    dump = sim.debug_step(None)
    orc = ref64.Oracle(ref64.fields_from(model.field))
    for e in range(B):
        states.oracle_step(orc, q[e], v[e], np.zeros(model.nv, np.float32), np.zeros(0, np.float32))
        for f in ("qfrc_smooth", "qacc"):
            a, b = dump.get(2, e, f), orc.get(f)
            assert np.max(np.abs(a - b)) < 1e-4 * max(1.0, np.max(np.abs(b))), (f, e)
