"""Rays go to the device in one copy up to 256 KB, in two beyond: a scan on either
side of the line gives what scans of its halves give."""
from __future__ import annotations

import numpy as np
import pytest

from mjmlx_hip import capi, scenes

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("rays", [2, 42, 170, 172, 400])  # 64 envs: 256 KB is between 170 and 172
def test_scan_equals_its_halves(rays):
    B, rng = 64, np.random.default_rng(rays)
    model = capi.Model(scenes.quadruped_xml())
    sim = capi.BatchedSim(model, B)
    sim.set_state(scenes.quadruped_initial_qpos(B, 1).astype(np.float32), np.zeros((B, model.nv), np.float32))
    p = rng.uniform(-0.3, 0.3, (B, rays, 3)).astype(np.float32) + np.float32([0, 0, 0.8])
    d = rng.normal(size=(B, rays, 3)).astype(np.float32)
    d /= np.linalg.norm(d, axis=2, keepdims=True)
    h = rays // 2
    whole = sim.raycast(p, d)
    halves = [sim.raycast(p[:, s].copy(), d[:, s].copy()) for s in (slice(0, h), slice(h, rays))]
    assert (whole[1] >= 0).mean() > 0.2
    for w, a, b in zip(whole, *halves):
        assert np.array_equal(w, np.concatenate([a, b], axis=1))
