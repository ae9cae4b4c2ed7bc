"""qM and its factor in a debug dump: nv x nv up to 64 dofs, whatever the kernels
store or skip."""
from __future__ import annotations

import numpy as np
import pytest

import ref64
from mjmlx_hip import capi, scenes

pytestmark = pytest.mark.gpu


# elliptic Newton models of 21 to 32 dofs solve without the factor; free bodies
# of 33 to 64 dofs store compact rows; the quadruped does neither
@pytest.mark.parametrize("scene", ["humanoid", "boxes6", "boxes8_newton", "quadruped"])
def test_mass_matrix_and_factor(scene):
    xml = {"humanoid": scenes.humanoid_xml(), "boxes6": scenes.boxes_xml(6, 106),
           "boxes8_newton": scenes.boxes_xml(8, 108, solver="Newton"), "quadruped": scenes.quadruped_xml()}[scene]
    model, B = capi.Model(xml), 5
    nv = model.nv
    rng = np.random.default_rng(3)
    q = np.tile(model.field("qpos0").astype(np.float32), (B, 1))
    q += rng.uniform(-0.02, 0.02, q.shape).astype(np.float32)
    v = np.zeros((B, nv), np.float32)
    sim = capi.BatchedSim(model, B)
    sim.set_state(q, v)
    dump = sim.debug_step(None)
    orc = ref64.Oracle(ref64.fields_from(model.field))
    for e in range(B):
        orc.set_state(q[e].astype(np.float64), v[e].astype(np.float64), np.zeros(nv), np.zeros(model.nu))
        orc.forward()
        M = orc.get("qM").reshape(nv, nv)
        M = np.tril(M) + np.tril(M, -1).T
        got = dump.get(1, e, "qM").reshape(nv, nv).astype(np.float64)
        assert np.max(np.abs(got - M)) < 1e-5 * np.max(np.abs(M))
        F = dump.get(1, e, "qLD").reshape(nv, nv).astype(np.float64)
        L = np.tril(F, -1) + np.eye(nv)
        assert np.max(np.abs(L.T @ (np.diag(F)[:, None] * L) - M)) < 1e-5 * np.max(np.abs(M))
