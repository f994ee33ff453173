"""The operator form's system and the calls around it (rf_operator.hip, rf_store.h):
a solve takes its loop bounds and addresses from the near store, so one without a
successful assembly is refused on the host; and the system is the assembled one,
whatever becomes of the state before the solve."""
import os
import subprocess

import numpy as np
import pytest

HERE = os.path.dirname(os.path.abspath(__file__))
ROOT = os.path.dirname(HERE)


def test_near_memory_holds_a_system_only_after_a_whole_assembly(tmp_path):
    """It holds a system only after a whole assembly, and grows on the simulation's GPU."""
    exe = tmp_path / "near_memory"
    subprocess.run(["g++", "-std=c++17", "-O1", "-Wall", "-Werror", "-I",
                    os.path.join(ROOT, "rigidfibers_amd", "csrc"),
                    os.path.join(HERE, "near_memory", "near_memory.cpp"), "-o", str(exe)], check=True)
    out = subprocess.run([str(exe)], capture_output=True, text=True, timeout=30)
    assert out.returncode == 0, out.stdout


def _sim(solver, M=1000, **kw):
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    pos, ori = cube(M, (M / 0.03) ** (1.0 / 3.0), min_dist=0.4, seed=M)
    params = Parameters(NUMBER_OF_FIBERS=M, GMRES_TOLERANCE=1e-8, BICGSTAB_TOLERANCE=1e-8)
    return pos, ori, Simulation(params, pos, ori, solver=solver, **kw)


@pytest.mark.gpu
@pytest.mark.parametrize("solver", ["gmres", "bicgstab", "gmres-ir"])
def test_solve_without_a_system_is_refused(solver):
    from rigidfibers_amd import _lib

    pos, ori, sim = _sim(solver)
    with sim:
        for _ in range(2):
            with pytest.raises(_lib.RfError) as err:
                sim.solve_system()
            assert err.value.code == _lib.RF_ERR_INVALID_ARGUMENT
        assert sim.solver_stats()["iterations"] == 0  # nothing ran
        sim.assemble_system()
        sim.solve_system()
        _, b, x = sim.system()
        assert sim.solver_stats()["converged"] and np.isfinite(x).all() and b.any()
        assert sim.step(0) == 0


@pytest.mark.gpu
@pytest.mark.parametrize("solver,integration", [("gmres", "numerical"), ("bicgstab", "analytical"),
                                                ("gmres-ir", "numerical")])
def test_the_state_moves_before_the_solve(solver, integration):
    """A solve after rf_set_state or rf_advance is of the assembled system: the same
    kernels on the same numbers from the same start (zero), so bit for bit."""
    def solution(move):
        pos, ori, sim = _sim(solver, integration=integration, initial_guess="zero")
        with sim:
            sim.assemble_system()
            move(sim, pos, ori)
            sim.solve_system()
            return sim.system()[1:]

    def overwrite(sim, pos, ori):
        sim.set_state(1.01 * pos, ori[::-1].copy())

    def advance(sim, pos, ori):
        sim.solve_system()
        sim.update_velocities()
        sim.update_fibers(True)
        sim.advance()

    b, x = solution(lambda *_: None)
    for move in (overwrite, advance):
        b1, x1 = solution(move)
        assert np.array_equal(b1, b) and np.array_equal(x1, x)


@pytest.mark.gpu
def test_noalloc_dump_forms_the_same_columns():
    """rf_get_system_noalloc forms the operator form's dense matrix 12 source fibers
    at a time (8 terms: 12 x 24 columns of 13 512 rows fill the 16 MiB staging
    buffer), the last range 11 of 563: bit for bit rf_get_system's, the diagonal
    blocks the identity."""
    import ctypes as C

    from rigidfibers_amd import _lib
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    M, N = 563, 8
    pos, ori = cube(M, (M / 0.05) ** (1.0 / 3.0), min_dist=0.4, seed=M)
    params = Parameters(NUMBER_OF_FIBERS=M, NUMBER_OF_TERMS_IN_FORCE_EXPANSION=N)
    with Simulation(params, pos, ori, integration="analytical") as sim:
        theta_bytes = 4 * M * M * N * (3 + 6 * (N - 1))
        assert sim.device_bytes() < theta_bytes  # the operator form
        sim.step(0)  # the matrix belongs to the state before the step
        A0, b0, x0 = sim.system(with_matrix=True)
        A1 = np.full((sim.n, sim.n), np.nan, dtype=np.float32, order="F")
        b1, x1 = np.full(sim.n, np.nan), np.full(sim.n, np.nan)
        _lib.check(sim._lib.rf_get_system_noalloc(sim._h, A1.ctypes.data_as(C.POINTER(C.c_float)),
                                                  b1.ctypes.data_as(C.POINTER(C.c_double)),
                                                  x1.ctypes.data_as(C.POINTER(C.c_double))))
    assert np.array_equal(A0, A1) and np.array_equal(b0, b1) and np.array_equal(x0, x1)
    for j in (0, 11, 12, 551, 552, 562):  # ends of ranges
        d = slice(24 * j, 24 * (j + 1))
        assert np.array_equal(A0[d, d], np.eye(24, dtype=np.float32))
    r = b0[:2400] - A0[:2400].astype(np.float64) @ x0
    assert np.linalg.norm(r) <= 1e-4 * np.linalg.norm(b0)
