"""Read-back of particles and grids (csrc/host_copy.h): bytes as loaded, where
the copy can go wrong: one particle, a count that is no multiple of the four
floats a thread stores, ranges that start anywhere, one element around a half
of the pinned buffer (1 400 000 particles) and more than its two halves."""
import numpy as np
import pytest

from ffengine import FluidSimulation

pytestmark = pytest.mark.gpu
HALF = 1400000


@pytest.mark.parametrize("n", [1, 5, HALF, HALF + 1, 2 * HALF + 3, 3 * HALF + 1])
def test_particles_read_back_as_loaded(n):
    print("read-back of", n, flush=True)
    rng = np.random.default_rng(n)
    pos = (0.1 + 0.8 * rng.random((n, 3), np.float32)).astype(np.float32)
    vel = rng.standard_normal((n, 3), np.float32)
    sim = FluidSimulation(16, 16, 16, 1.0 / 16)
    for a in range(0, n, 200000):  # the reference's load queue reorders loads of 208333 particles and more
        b = min(a + 200000, n)
        sim.load_marker_particle_data(b - a, pos[a:b].tobytes(), vel[a:b].tobytes())
    sim.initialize()
    for a, b in ((0, n), (min(3, n), n), (n // 2, max(n // 2, n - 2)), (n, n)):
        assert sim.get_marker_particle_position_data_range(a, b) == pos[a:b].tobytes()
        assert sim.get_marker_particle_velocity_data_range(a, b) == vel[a:b].tobytes()
    assert sim.get_marker_particle_position_data() == pos.tobytes()
    for bad in ((-1, n), (0, n + 1), (n, n - 1)):
        with pytest.raises(Exception):
            sim.get_marker_particle_position_data_range(*bad)


@pytest.mark.parametrize("n3", [(3, 3, 3), (255, 129, 130)])  # the larger: 17 MB, just over a half
def test_solid_sdf_reads_back_as_set(n3):
    shape = tuple(a + 1 for a in n3[::-1])
    phi = np.random.default_rng(1).standard_normal(shape).astype(np.float32)
    sim = FluidSimulation(*n3, 1.0 / max(n3))
    sim.set_solid_phi(phi)
    sim.initialize()
    assert sim.get_solid_sdf().tobytes() == phi.tobytes()


def test_read_back_from_two_threads():
    """Positions in one thread and velocities in another, of one simulation and
    at once: each gets its own bytes."""
    import threading
    n = HALF + 1
    rng = np.random.default_rng(n)
    pos = (0.1 + 0.8 * rng.random((n, 3), np.float32)).astype(np.float32)
    vel = rng.standard_normal((n, 3), np.float32)
    sim = FluidSimulation(16, 16, 16, 1.0 / 16)
    for a in range(0, n, 200000):
        b = min(a + 200000, n)
        sim.load_marker_particle_data(b - a, pos[a:b].tobytes(), vel[a:b].tobytes())
    sim.initialize()
    print("read-back of", n, "by two threads", flush=True)
    wrong = []

    def read(get, want):
        for size in (5, 1000, n // 3, n):  # ascending: the pinned buffer grows under way
            if get(0, size) != want[:size].tobytes():
                wrong.append((get.__name__, size))

    team = [threading.Thread(target=read, args=a) for a in
            ((sim.get_marker_particle_position_data_range, pos), (sim.get_marker_particle_velocity_data_range, vel))]
    for t in team:
        t.start()
    for t in team:
        t.join()
    assert not wrong


def test_a_missing_buffer_is_an_error():
    """A grid read into no buffer fails with an error, as the copy into it did,
    and the simulation goes on."""
    from ctypes import byref, c_int, c_void_p
    from ffengine.ffengine import ffengine as lib
    sim = FluidSimulation(16, 16, 16, 1.0 / 16)
    sim.load_marker_particle_data(1, np.full(3, 0.5, np.float32).tobytes(), np.zeros(3, np.float32).tobytes())
    sim.initialize()
    for name in ("pressure_grid", "liquid_sdf", "solid_sdf"):
        err = c_int(1)
        f = getattr(lib, "FluidSimulation_get_%s_data" % name)
        f.argtypes, f.restype = [c_void_p, c_void_p, c_void_p], None
        f(sim(), None, byref(err))
        assert err.value == 0, name
    assert sim.get_pressure_grid().shape == (16, 16, 16)
