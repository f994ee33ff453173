"""The iterative solvers' start on the device (rigidfibers_amd/csrc/rf_linalg.hip):
a right-hand side of zeros, a tolerance that x = 0 meets, an iteration limit of
the one step, and a right-hand side that is not finite, in one workgroup (up to
8192 unknowns) and in several (546 fibers of 5 terms are 8190 unknowns, 547 are
8205).  The outcomes are exact: no tolerance but the solver's own."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


def _sim(M, solver, coincident=False, force=(0.0, 0.0, -1.0), **kw):
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    pos, ori = cube(M, (M / 0.03) ** (1.0 / 3.0), min_dist=0.4, seed=M)
    if coincident:
        pos[3:6], ori[3:6] = pos[0:3], ori[0:3]
    params = Parameters(NUMBER_OF_FIBERS=M, NUMBER_OF_TERMS_IN_FORCE_EXPANSION=5, GMRES_RESTART=10, **kw)
    return pos, ori, Simulation(params, pos, ori, solver=solver, integration="numerical", external_force=force)


@pytest.mark.parametrize("M", [20, 546, 547])
@pytest.mark.parametrize("solver", ["gmres", "bicgstab", "gmres-ir"])
def test_solver_starts(M, solver):
    from rigidfibers_amd import _lib

    _, _, sim = _sim(M, solver, force=(0.0, 0.0, 0.0))
    with sim:  # no force: nothing moves
        for t in range(2):
            assert sim.step(t) == 0
        _, b, x = sim.system()
        stats = sim.solver_stats()
    assert not b.any() and not x.any() and stats["converged"] and stats["iterations"] == 0

    _, _, sim = _sim(M, solver, GMRES_TOLERANCE=2.0, BICGSTAB_TOLERANCE=2.0)
    with sim:  # x = 0 has the relative residual 1
        assert sim.step(0) == 0
        _, b, x = sim.system()
        stats = sim.solver_stats()
    assert b.any() and not x.any() and stats["converged"] and stats["iterations"] == 0
    assert abs(stats["relative_residual"] - 1.0) < 1e-12

    _, _, sim = _sim(M, solver, GMRES_TOLERANCE=1e-14, BICGSTAB_TOLERANCE=1e-14, GMRES_MAX_ITERATIONS=1,
                     BICGSTAB_MAX_ITERATIONS=1)
    with sim:
        assert sim.step(0) == _lib.RF_WARN_NOT_CONVERGED
        stats = sim.solver_stats()
    assert not stats["converged"] and stats["iterations"] == 1 and 1e-14 < stats["relative_residual"] < 1.0

    pos, ori, sim = _sim(M, solver, coincident=True)
    with sim:  # fails twice the same way, and the state stays where it was
        for _ in range(2):
            with pytest.raises(_lib.RfError) as err:
                sim.step(0)
            assert err.value.code == _lib.RF_ERR_NONFINITE
        p, o = sim.state()
        with pytest.raises(_lib.RfError):
            sim.advance()
    assert np.array_equal(p, pos) and np.array_equal(o, ori)
