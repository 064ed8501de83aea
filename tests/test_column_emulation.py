"""The column MIC(0) sweeps (csrc/column_sweep.h) emulated on the CPU.

tests/emu/column_emu.cpp compiles the GPU sweep's own body with g++ and runs
its lanes as fibers, the workgroups at once.  Each case applies the
preconditioner in FP64, FP32 and FP64 again over the same exchange words and
must equal, bit for bit, the oracle's serial sweeps (FP64, pcgsolver.h:211-241)
and a hyperplane-vectorised FP32 restatement.  The emulation gives a ring value
only the ordering that the sweep asks for, and checks that every buffer lies
inside its array.  Sides around the multiples of a column's 16 x 8 lines and of
a tile's two columns, more steps than the ring holds, and columns and tiles
without rows between ones with rows.
"""
import os
import shutil
import subprocess

import numpy as np
import pytest

import oracle_lib as O
from test_pencil_emulation import _mic_sweeps, _records

HERE = os.path.dirname(os.path.abspath(__file__))


@pytest.fixture(scope="module")
def emulator(tmp_path_factory):
    if shutil.which("g++") is None:
        pytest.skip("g++ is not installed")
    exe = str(tmp_path_factory.mktemp("emu") / "column_emu")
    subprocess.run(["g++", "-std=c++20", "-O1", "-g", "-ffp-contract=off", "-fsanitize=undefined",
                    "-fno-sanitize-recover=all", "-pthread", os.path.join(HERE, "emu", "column_emu.cpp"), "-o", exe],
                   check=True)
    return exe


def _system(kind, n3):
    from test_gpu_columns import _liquid  # (that module is GPU-marked)
    rng = np.random.default_rng(sum(n3) + len(kind))
    ni, nj, nk = n3
    dx = 1.0 / max(n3)
    phi = _liquid(kind, n3, rng)
    weights = O.face_weights(n3, O.solid_box_phi(n3, dx))
    uvw = [rng.standard_normal(s).astype(np.float32) for s in ((nk, nj, ni + 1), (nk, nj + 1, ni), (nk + 1, nj, ni))]
    sysm = O.pressure_system(n3, dx, 1.0 / 120.0, uvw, weights, phi)
    return sysm, rng.standard_normal(len(sysm["rows"]))


def _run(exe, tmp_path, n3, sysm, r, what):
    m = len(r)
    cell_row = np.full(int(np.prod(n3)), -1, np.int32)
    cell_row[sysm["rows"]] = np.arange(m, dtype=np.int32)
    fin, fout = tmp_path / "in.bin", tmp_path / "out.bin"
    with open(fin, "wb") as f:
        f.write(np.array([*n3, m], np.int32).tobytes())
        f.write(cell_row.tobytes())
        for a in (r, *_records(sysm)):
            f.write(np.ascontiguousarray(a, np.float64).tobytes())
    subprocess.run([exe, str(fin), str(fout), what], check=True, timeout=300)
    return np.fromfile(fout, np.float64).reshape(2, m) if what != "lost" else None


def _check(emulator, tmp_path, n3, kind, what):
    sysm, r = _system(kind, n3)
    z64, z32 = _run(emulator, tmp_path, n3, sysm, r, what)
    assert np.array_equal(z64.view(np.uint64), O.apply_mic0(sysm, r).view(np.uint64))
    want = _mic_sweeps(sysm, n3, r, np.float32)
    assert np.array_equal(z32.astype(np.float32).view(np.uint32), want.view(np.uint32))


@pytest.mark.parametrize("n3,kind", [((3, 3, 3), "full")] + [
    (n3, kind) for n3 in ((9, 16, 33), (40, 33, 8), (7, 40, 20), (31, 15, 47))
    for kind in ("full", "scattered", "islands", "layer")])
def test_column_sweeps_emulated_bitexact(emulator, tmp_path, n3, kind):
    _check(emulator, tmp_path, n3, kind, "plain")


def test_a_lost_workgroup_ends_the_launch(emulator, tmp_path):
    """A wait for a workgroup that never runs ends at the limit: the launch
    finishes with the error raised."""
    n3 = (9, 40, 33)
    sysm, r = _system("full", n3)
    _run(emulator, tmp_path, n3, sysm, r, "lost")
