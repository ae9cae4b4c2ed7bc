"""Where a step's workspaces live: the placement chosen at creation, its number
and what selects it again."""
from __future__ import annotations

import re

import numpy as np
import pytest

from mjmlx_hip import capi, scenes
from test_reference_models import model_xml
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


def _side_by_side(xml, n):
    """n copies of a scene's bodies and actuators, 3 m apart."""
    xml = re.sub(r"<contact>.*?</contact>", "", xml, flags=re.S)  # excludes name the bodies
    a, b = xml.index("<body"), xml.index("</worldbody>")
    c, d = xml.index("<actuator>") + len("<actuator>"), xml.index("</actuator>")
    name = lambda t, k: re.sub(r'\b(name|joint|site)="([^"]+)"', rf'\1="\2_{k}"', t)  # noqa: E731
    x = re.compile(r'(<body[^>]*? pos=")([-\d.]+)')
    bodies = "".join(x.sub(lambda m: f"{m[1]}{float(m[2]) + 3 * k}", name(xml[a:b], k), count=1) for k in range(n))  # noqa: B023
    return xml[:a] + bodies + xml[b:c] + "".join(name(xml[c:d], k) for k in range(n)) + xml[d:]


def _model(name):
    if name == "tree54":
        return model_xml("high_dof_tree")
    kind, n = name[:-1], int(name[-1])
    if kind == "boxes":
        return scenes.boxes_xml(n, 100 + n)
    if kind == "quadrupeds":
        return _side_by_side(scenes.quadruped_xml(self_collision=False), n)
    return _side_by_side(scenes.humanoid_xml(self_collision=False), n)


LDS, DEVICE = 3, 1  # at most four envs of these per CU: the whole register file


# A model of more than 32 dofs keeps LDS unless another placement was measured to
# be faster for its kind: free bodies go to small workspaces or device memory,
# articulated models to small workspaces, to device memory only from four times
# its rounds on, and with elliptic cones under Newton they stay.
@pytest.mark.parametrize("name,B,want", [
    ("boxes6", 300, LDS), ("boxes6", 600, COMPACT), ("boxes6", 2100, DEVICE), ("boxes8", 4096, DEVICE),
    ("quadrupeds2", 300, LDS), ("quadrupeds2", 1100, COMPACT), ("quadrupeds2", 2100, LDS), ("quadrupeds2", 4096, LDS),
    ("quadrupeds3", 1100, LDS), ("quadrupeds3", 4096, DEVICE), ("tree54", 300, COMPACT), ("tree54", 1100, DEVICE),
    ("humanoids2", 300, LDS), ("humanoids2", 1100, LDS)])
def test_default_placement(name, B, want):
    assert capi.BatchedSim(capi.Model(_model(name)), B).variant() == want


def test_dense_rows_keep_the_given_placement(monkeypatch):
    monkeypatch.setenv("MJMLX_HIP_DENSE_ROWS", "1")
    assert capi.BatchedSim(capi.Model(scenes.boxes_xml(6, 106)), 2100).variant() == LDS


@pytest.mark.parametrize("graph", [False, True])
def test_captured_step_follows_the_variant(graph):
    """A learned control step captured as a graph is captured again when the
    variant changes, also where only small workspaces go. Both variants give the
    same bits, so the time tells: 8 boxes, 600 envs take about 2.5 times as long
    in full-size LDS workspaces."""
    n, B = 8, 600
    model = capi.Model(scenes.boxes_xml(n, 108))
    rng = np.random.default_rng(0)
    sim = capi.BatchedSim(model, B)
    assert sim.variant() == COMPACT
    sim.set_state(_states(model, n, B, np.zeros(B, bool), rng), np.zeros((B, 6 * n), np.float32))
    sim.set_warmstart_mlp(capi.MLP(sim.feature_dim(), 64, 6 * n, seed=1))
    assert sim.set_warmstart_mode(2) == 0
    sim.set_graph(graph)
    ms = []
    for v in (COMPACT, 3):
        assert sim.variant() == v or sim.set_variant(v)
        t = []
        for _ in range(6):
            sim.step(None, 2)
            sim.sync()
            t.append(sim.last_step_ms())
        ms.append(float(np.median(t[2:])))
    print(f"graph {graph}: small workspaces {ms[0]:.3f} ms, full-size LDS {ms[1]:.3f}")
    assert ms[1] > 1.6 * ms[0]


def test_captured_step_follows_the_network():
    """A network freed and another made, which may get the first one's address."""
    B = 64
    model = capi.Model(scenes.quadruped_xml())
    out = []
    for graph in (False, True):
        sim = capi.BatchedSim(model, B)
        sim.set_graph(graph)
        for seed, width in ((1, 64), (2, 128), (3, 64)):
            net = capi.MLP(sim.feature_dim(), width, model.nv, seed=seed)
            net.set_normalization(out_std=np.full(model.nv, 20.0))
            sim.set_warmstart_mlp(net)
            assert sim.set_warmstart_mode(2) == 0
            for _ in range(4):
                sim.step(None, 2)
            out.append((*sim.state(), sim.stats()["niter"]))
            sim.set_warmstart_mlp(None)
            del net
    for a, b in zip(out[:3], out[3:]):
        for x, y in zip(a, b):
            assert np.array_equal(x, y)
