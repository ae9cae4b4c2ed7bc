"""The qM solve of the 64-lane kernels is no less exact than the tree factor.

qacc_smooth against the FP64 solution of the same FP32 problem (the kernel's own
qM and qfrc_smooth): the RMS over many states may not exceed that of the 32-lane
kernels, which factor qM level by level at every size. Elliptic chains, whose
64-lane kernels solve in registers beyond 20 dofs. The two roundings of a state
are independent draws of one size, so the ratio of two RMS over N states
spreads by about 1 / sqrt(N), 2.2 % here: 4.5 of them."""
from __future__ import annotations

import numpy as np
import pytest

from mjmlx_hip import capi
from test_gpu_elliptic_regs import _elliptic

pytestmark = pytest.mark.gpu

N = 2000


def _rms(model, variant, q, v):
    nv = model.nv
    sim = capi.BatchedSim(model, N)
    assert sim.set_variant(variant)
    sim.set_state(q, v)
    dump = sim.debug_step(None)
    get = lambda k, n: np.stack([dump.get(2, e, k)[:n] for e in range(N)]).astype(np.float64)  # noqa: E731
    M, f, x = get("qM", nv * nv).reshape(N, nv, nv), get("qfrc_smooth", nv), get("qacc_smooth", nv)
    t = np.linalg.solve(M, f[..., None])[..., 0]
    e = np.linalg.norm(x - t, axis=1) / np.linalg.norm(t, axis=1)
    return float(np.sqrt(np.mean(e * e)))


@pytest.mark.parametrize("nv", [12, 17, 18, 19, 20, 21, 27, 32])
def test_no_less_exact_than_the_tree_factor(nv):
    model = capi.Model(_elliptic(nv, "limit"))
    rng = np.random.default_rng(nv)
    q, v = (rng.uniform(-0.5, 0.5, (N, nv)).astype(np.float32) for _ in range(2))
    regs, tree = _rms(model, 0, q, v), _rms(model, 5, q, v)
    print(f"{nv} dofs: 64 lanes {regs:.2e}, tree factor {tree:.2e}, ratio {regs / tree:.3f}")
    assert regs <= 1.1 * tree
