"""The FP64 curvature at every size of angle between neighbouring directors, on
both sides of where its arc cosine changes form (1/4, 60 degrees) and up to
half a turn: both FP64 paths equal the oracle bitwise, angles of one size in a
wave and of all sizes in one."""
import numpy as np
import pytest

from elasticapp_amd import FP64
from tests.gpu_helpers import STATE, device_block, oracle_system, random_workload

pytestmark = pytest.mark.gpu

ANGLES = [0.0, 1e-9, 2e-5, 1e-3, 0.24999, 0.25001, 1.0471, 1.0473, 1.6, 2.6, 3.1, 3.1415926]


@pytest.mark.parametrize("angle", ANGLES + ["all"])
def test_curvature_equals_the_oracle(angle):
    wl = random_workload(0, 0, 0, seed=77, lengths=[64, 30, 100], vstd=1e-4)
    rng = np.random.default_rng(5)
    for st in wl.states:
        n = st["Director"].shape[1]
        q = st["Director"][:, 0].reshape(3, 3)
        out = np.empty((9, n))
        for k in range(n):
            out[:, k] = q.ravel()
            a = rng.choice(ANGLES) if angle == "all" else angle
            u = rng.normal(size=3)
            u /= np.linalg.norm(u)
            U = np.array([[0, -u[2], u[1]], [u[2], 0, -u[0]], [-u[1], u[0], 0]])
            q = (np.eye(3) + np.sin(a) * U + (1 - np.cos(a)) * U @ U) @ q
        st["Director"] = out
    sysm = oracle_system(wl, variant="devmath")
    fused, plain = device_block(wl), device_block(wl)
    for n in (1, 3):
        with np.errstate(all="ignore"):
            sysm.step(1e-9, n)
        fused.set_rod_dt(1e-9)
        fused.step_fused(n, FP64)
        plain.step(1e-9, n)
        for r in range(3):
            for tag in STATE:
                c = sysm.rod_field(r, tag)
                assert np.array_equal(fused.get_rod(tag, r), c, equal_nan=True), (n, r, tag)
                assert np.array_equal(plain.get_rod(tag, r), c, equal_nan=True), (n, r, tag)
