"""FP64 divisions and square roots without their special cases, and the full
ones in waves where an operand does not allow that: every state the two forms
could part at equals the oracle's, bitwise, on the fused path and on the
op-by-op one: exact zeros, values at both ends of the exponent range and
denormal ones (fronts that have just reached an element), lengths outside the
plain forms' range, rods that overflow, and ordinary rods beside each in one
wave."""
import numpy as np
import pytest

from elasticapp_amd import FP64
from tests.gpu_helpers import STATE, device_block, oracle_system, random_workload

pytestmark = pytest.mark.gpu


def _still(st):
    st["Velocity"][:] = 0.0
    st["AngularVelocity"][:] = 0.0
    st["ReferenceCurvature"][:] = 0.0
    st["ReferenceShearStretchStrain"][:] = 0.0


def _scaled(st, factor):
    for tag in ("Position", "ReferenceElementLength", "ReferenceVoronoiLength"):
        st[tag] = st[tag] * factor


def _change(kind, st, rng):
    if kind == "zero":
        _still(st)
    elif kind == "tiny":
        # straight, unstrained, each value of its own scale down to denormals
        _still(st)
        st["Velocity"] = rng.normal(size=st["Velocity"].shape) * 10.0 ** rng.uniform(-323, -200, st["Velocity"].shape)
        st["AngularVelocity"] = rng.normal(size=st["AngularVelocity"].shape) * 10.0 ** rng.uniform(
            -323, -200, st["AngularVelocity"].shape)
    elif kind == "front":
        # at rest but for one element in the middle: what leaves it underflows on its way
        _still(st)
        st["AngularVelocity"][1, st["AngularVelocity"].shape[1] // 2] = 1e-3
    elif kind == "short":
        _scaled(st, 1e-32)   # lengths below 2^-100
    elif kind == "long":
        _scaled(st, 1e33)    # and above 2^100
    elif kind == "overflow":
        st["Velocity"][0, 1] = 1e180
        st["AngularVelocity"][2, 0] = 1e170
    elif kind == "nonfinite":
        st["Velocity"][1, 0] = np.inf
        st["AngularVelocity"][0, -1] = np.nan


@pytest.mark.parametrize("kind", ["zero", "tiny", "front", "short", "long", "overflow", "nonfinite"])
def test_both_forms_round_like_the_oracle(kind):
    rng = np.random.default_rng(11)
    wl = random_workload(0, 0, 0, seed=601, forces=kind in ("zero", "short"), lengths=[20, 50, 200, 7, 90, 64])
    for r in (0, 2, 3):
        _change(kind, wl.states[r], rng)
    sysm = oracle_system(wl, variant="devmath")
    fused, plain = device_block(wl), device_block(wl)
    for n in (1, 2, 25):
        with np.errstate(all="ignore"):
            sysm.step(wl.dt, n)
        fused.step_fused(n, FP64)
        plain.step(wl.dt, n)
        for r in range(len(wl.n_elems)):
            for tag in STATE:
                c = sysm.rod_field(r, tag)
                assert np.array_equal(fused.get_rod(tag, r), c, equal_nan=True), (n, r, tag)
                assert np.array_equal(plain.get_rod(tag, r), c, equal_nan=True), (n, r, tag)
    if kind in ("overflow", "nonfinite"):
        assert fused.check_finite()[[0, 2, 3]].all() and not fused.check_finite()[[1, 4, 5]].any()


@pytest.mark.parametrize("scale", [1e-320, 1e-316, 1e-312, 1e-306])
def test_denormal_numerators_between_ordinary_ones(scale):
    """A stretched straight rod that spins by denormal rates: in its divisions
    by the dilatation every numerator is zero, ordinary, or below 2^-1042, where
    a plain division loses the last unit."""
    from elasticapp_amd import straight_rod_state

    rng = np.random.default_rng(5)
    wl = random_workload(0, 0, 0, seed=602, forces=False, lengths=[60, 100])
    for r, n in enumerate(wl.n_elems):
        st = straight_rod_state(n, 0.02, 1.0, [0.0, 0.0, 0.0], [1.0, 0.0, 0.0], [0.0, 0.0, 1.0], 1000.0, 1e6, 4e5, 0.1, 0.1)
        st["Position"] = st["Position"] * 1.3
        st["Velocity"][0] = rng.normal(size=n + 1)
        st["AngularVelocity"] = scale * rng.normal(size=(3, n))
        wl.states[r] = st
    sysm = oracle_system(wl, variant="devmath")
    fused, plain = device_block(wl), device_block(wl)
    for n in (1, 2, 10):
        sysm.step(wl.dt, n)
        fused.step_fused(n, FP64)
        plain.step(wl.dt, n)
        for r in range(len(wl.n_elems)):
            for tag in STATE:
                c = sysm.rod_field(r, tag)
                assert np.array_equal(fused.get_rod(tag, r), c), (n, r, tag)
                assert np.array_equal(plain.get_rod(tag, r), c), (n, r, tag)
