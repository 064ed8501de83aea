"""The MIC(0) application in the column layout (csrc/kernels_column.hip, the
solver's schedule) against the oracle's serial sweeps (FP64) and a
hyperplane-vectorised FP32 restatement, bit for bit, where its split into
columns of 16 x 8 lines, tiles of two of them and rounds of steps can go
wrong: sides around the multiples of those, one line of cells, columns and
tiles without rows between ones with rows, scattered rows."""
import numpy as np
import pytest

import oracle_lib as O
from ffengine import kernels as K
from test_gpu_kernels import _mic_sweeps, same_bits, say

pytestmark = pytest.mark.gpu


def _liquid(kind, n3, rng):
    ni, nj, nk = n3
    k, j, i = np.meshgrid(np.arange(nk), np.arange(nj), np.arange(ni), indexing="ij")
    if kind == "full":
        wet = np.ones((nk, nj, ni), bool)
    elif kind == "scattered":
        wet = rng.random((nk, nj, ni)) < 0.3
    elif kind == "islands":  # two blocks with empty columns and tiles between
        wet = ((j < 5) & (k < 6)) | ((j >= nj - 6) & (k >= nk - 7) & (i > ni // 2))
    else:  # "layer": every column spans few hyperplanes, at different heights
        wet = (j + 2 * k) // 3 % 11 == i % 11
    return np.where(wet, np.float32(-0.4), np.float32(0.3)).astype(np.float32) / max(n3)


@pytest.mark.parametrize("kind", ["full", "scattered", "islands", "layer"])
@pytest.mark.parametrize("n3", [(3, 3, 3), (5, 17, 9), (9, 16, 33), (40, 33, 8), (31, 15, 47), (130, 18, 34), (7, 70, 20)])
def test_column_sweeps_bitexact(n3, kind):
    rng = np.random.default_rng(sum(n3) + len(kind))
    dx, dt = 1.0 / max(n3), 1.0 / 120.0
    ni, nj, nk = n3
    phi = _liquid(kind, n3, rng)
    weights = O.face_weights(n3, O.solid_box_phi(n3, dx))
    uvw = [rng.standard_normal(s).astype(np.float32) for s in ((nk, nj, ni + 1), (nk, nj + 1, ni), (nk + 1, nj, ni))]
    sysm = O.pressure_system(n3, dx, dt, uvw, weights, phi)
    m = len(sysm["rows"])
    if m == 0:
        pytest.skip("no rows")
    r = rng.standard_normal(m)
    say(f"column sweeps {n3} {kind}: {m} rows")
    z = K.mic0_apply(n3, dx, dt, uvw, weights, phi, r, precision=0, schedule=2)
    assert same_bits(z, O.apply_mic0(sysm, r))
    f = K.mic0_apply(n3, dx, dt, uvw, weights, phi, r, precision=1, schedule=2)
    # the call adds the widened FP32 result to zeros: -0 comes back as +0
    assert same_bits(f.astype(np.float32), _mic_sweeps(sysm, n3, r, np.float32) + np.float32(0))


@pytest.mark.parametrize("schedule", [2, 3, 0], ids=["columns", "bands-device-check", "hyperplanes"])
@pytest.mark.parametrize("value", [np.inf, -np.inf, np.nan, 1e300])
@pytest.mark.parametrize("n3", [(9, 16, 33), (31, 15, 47), (40, 40, 70)])
def test_non_finite_values_stay_in_their_body(n3, value, schedule):
    """A value that is, or in the sweeps or as a float becomes, infinite or NaN
    changes the rows that depend on it and no others: the other of two bodies of
    liquid, a cell apart along the lines they share, keeps its bits, and in its
    own body it goes where the serial sweeps take it."""
    ni, nj, nk = n3
    rng = np.random.default_rng(sum(n3))
    k, j, i = np.meshgrid(np.arange(nk), np.arange(nj), np.arange(ni), indexing="ij")
    phi = np.where(i != ni // 2, np.float32(-0.4), np.float32(0.3)).astype(np.float32) / max(n3)
    weights = O.face_weights(n3, O.solid_box_phi(n3, 1.0 / max(n3)))
    uvw = [rng.standard_normal(s).astype(np.float32) for s in ((nk, nj, ni + 1), (nk, nj + 1, ni), (nk + 1, nj, ni))]
    args = n3, 1.0 / max(n3), 1.0 / 120.0, uvw, weights, phi
    sysm = O.pressure_system(*args)
    m = len(sysm["rows"])

    def agree(got, want):
        finite = np.isfinite(want)
        assert np.array_equal(np.isfinite(got), finite)
        assert np.array_equal(got, want, equal_nan=True)
        assert same_bits(got[finite], want[finite])

    for at in (0, m - 1):  # in the one body, ahead of the other in the forward sweep, and in the other one
        r = rng.standard_normal(m)
        r[at] = value
        say(f"row {at} of {m} is {value}, {n3} schedule {schedule}")
        want = O.apply_mic0(sysm, r)
        assert np.isfinite(want).sum() >= m // 3
        agree(K.mic0_apply(*args, r, precision=0, schedule=schedule), want)
        with np.errstate(all="ignore"):
            want = _mic_sweeps(sysm, n3, r, np.float32) + np.float32(0)
            got = K.mic0_apply(*args, r, precision=1, schedule=schedule).astype(np.float32)
        assert m // 3 <= np.isfinite(want).sum() < m
        agree(got, want)


def test_a_system_without_divergence_has_its_factor():
    """The matrix and its factor do not depend on the velocities: with none, so
    that there is nothing to solve, the factor and its application are the
    oracle's all the same."""
    n3, dx = (20, 18, 19), 1.0 / 20
    rng = np.random.default_rng(1)
    phi = _liquid("scattered", n3, rng)
    weights = O.face_weights(n3, O.solid_box_phi(n3, dx))
    ni, nj, nk = n3
    uvw = [np.zeros(s, np.float32) for s in ((nk, nj, ni + 1), (nk, nj + 1, ni), (nk + 1, nj, ni))]
    args = n3, dx, 1.0 / 120.0, uvw, weights, phi
    sysm = O.pressure_system(*args)
    r = rng.standard_normal(len(sysm["rows"]))
    say(f"no divergence: {len(r)} rows")
    assert not sysm["rhs"].any()
    assert same_bits(K.pressure_system(*args)["invdiag"], sysm["invdiag"])
    for schedule in (2, 4, 3, 0):
        assert same_bits(K.mic0_apply(*args, r, precision=0, schedule=schedule), O.apply_mic0(sysm, r))
        got = K.mic0_apply(*args, r, precision=1, schedule=schedule).astype(np.float32)
        assert same_bits(got, _mic_sweeps(sysm, n3, r, np.float32) + np.float32(0))


@pytest.mark.parametrize("precision", ["fp64", "fp32-preconditioner", "mixed", "mixed-reliable"])
def test_every_sweep_is_timed(precision):
    """The kernel timing of the MIC(0) application counts every sweep of a solve:
    two an iteration and two before the first, but for a solve's last iteration
    (mixed: each inner solve's), which runs the forward one; a replaced residual
    (mixed-reliable) runs the forward one again."""
    from ctypes import byref, c_double, c_int, c_longlong, c_void_p
    from ffengine import scenes
    from ffengine.ffengine import ffengine as lib
    from test_gpu_engine import make_gpu
    lib.FluidSimulation_enable_kernel_timing.argtypes = [c_void_p, c_int, c_void_p]
    lib.FluidSimulation_get_kernel_timing.argtypes = [c_void_p, c_int, c_void_p, c_void_p, c_void_p]
    sim = make_gpu(24, scenes.dam_break_particles(24, seed=3), precision=precision, tol=1e-8)
    ok = c_int()
    lib.FluidSimulation_enable_kernel_timing(sim(), 1, byref(ok))
    assert ok.value
    sim.step(1.0 / 240.0)
    its = sim.get_last_pressure_solve_stats()["iterations"]
    ms, launches = c_double(), c_longlong()
    lib.FluidSimulation_get_kernel_timing(sim(), 7, byref(ms), byref(launches), byref(ok))
    say(f"{precision}: {its} iterations, {launches.value} sweeps")
    assert ok.value and its > 1 and ms.value > 0
    if precision in ("fp64", "fp32-preconditioner"):
        assert launches.value == 2 * its + 1
    else:
        assert 2 * its + 1 < launches.value <= 4 * its


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_two_simulations_at_once(precision):
    """Two threads, each with a simulation of its own: their sweeps wait on the
    device for their own tiles only, and each frame is the one it is alone."""
    import threading
    from ffengine import scenes
    from test_gpu_engine import gpu_particles, make_gpu
    sizes = (33, 48)

    def run(n, out):
        sim = make_gpu(n, scenes.dam_break_particles(n, seed=n), precision=precision, tol=1e-8)
        for _ in range(3):
            sim.update(1.0 / 60.0)
        out[n] = [a.copy() for a in gpu_particles(sim)]

    alone, together = {}, {}
    for n in sizes:
        run(n, alone)
    say(f"{precision}: two simulations at once")
    team = [threading.Thread(target=run, args=(n, together)) for n in sizes]
    for t in team:
        t.start()
    for t in team:
        t.join()
    for n in sizes:
        for a, b in zip(alone[n], together[n]):
            assert np.array_equal(a.view(np.uint32), b.view(np.uint32)), n
