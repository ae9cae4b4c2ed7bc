"""The register routines of small Newton models with elliptic cones (the qM solve
and the Newton direction; pyramidal models keep the workspace's factors), at the
edges of their sizes. A chain under ``cone="elliptic"`` without contacts takes
them for the same constraint rows as a pyramidal one, so the problems, bounds
and reasons are those of test_gpu_newton_regs.py and test_gpu_smooth_regs.py."""
from __future__ import annotations

import pytest

import states
import test_gpu_humanoid as humanoid
import test_gpu_newton_regs as newton
import test_gpu_smooth_regs as smooth
from mjmlx_hip import capi, scenes
from test_robustness_sweep import chain_xml

pytestmark = pytest.mark.gpu

SIZES = [1, 2, 4, 5, 19, 20, 21, 31, 32]


def _elliptic(nv, cfg):
    xml = chain_xml(nv, cfg)
    assert "<option " in xml and "cone=" not in xml
    return xml.replace("<option ", '<option cone="elliptic" ', 1)


@pytest.mark.parametrize("cfg", ["limit", "floss"])
@pytest.mark.parametrize("nv", SIZES)
def test_direction(nv, cfg, monkeypatch):
    monkeypatch.setattr(newton, "chain_xml", _elliptic)
    newton.test_direction_reaches_the_minimum(nv, cfg)


@pytest.mark.parametrize("nv", SIZES)
def test_smooth(nv, monkeypatch):
    monkeypatch.setattr(smooth, "chain_xml", _elliptic)
    smooth.test_chain(nv)


@pytest.mark.parametrize("variant", [0, 1, 2, 3])
def test_register_budgets(variant):
    """Humanoids under every register budget of the 64-lane kernels and from device
    memory (168 VGPRs: contacts read per evaluation, factors in the workspace), to
    the bars of the humanoid's parity test."""
    model = capi.Model(scenes.humanoid_xml())
    B = 24
    q, qv, qa, ctrl, orc = humanoid._states(model, B, 4)
    sim = capi.BatchedSim(model, B)
    assert sim.set_variant(variant)
    sim.set_state(q, qv)
    sim.set_qacc_warmstart(qa)
    dump = sim.debug_step(ctrl)
    st = sim.stats()
    assert not (st["status"] & ~3).any() and st["ncon"].sum() > B // 2
    for e in range(B):
        states.oracle_step(orc, q[e], qv[e], qa[e], ctrl[e])
        eq, ef = states.qacc_force_errors(orc, dump.get(2, e, "qacc"), dump.get(2, e, "efc_force"), st["nefc"][e])
        assert eq < 1e-4 and (ef or 0.0) < 1e-4, (e, eq, ef)
