"""The register routines of small Newton models with elliptic cones (the qM solve
and the Newton direction; pyramidal models keep the workspace's factors), at the
edges of their sizes. A chain under ``cone="elliptic"`` without contacts takes
them for the same constraint rows as a pyramidal one, so the problems, bounds
and reasons are those of test_gpu_newton_regs.py and test_gpu_smooth_regs.py."""
from __future__ import annotations

import pytest

import test_gpu_newton_regs as newton
import test_gpu_smooth_regs as smooth
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
