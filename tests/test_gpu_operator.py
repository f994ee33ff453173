"""The iterative solvers' operator form (rigidfibers_amd/csrc/rf_operator.hip):
large suspensions under matrix_format "auto" form the far pairs' kernel values in
each product; "theta" stores every pair.  Right-hand side and solution against
the FP64 oracle's rows of six target fibers (b, like the stored form's, is off by
the FP32 rounding of the near pairs' sums: within 4e-6 of its largest entry, the
solution's residual likewise), the state and velocities after a second step
against the stored form's run, to 1e-6 at a solver tolerance of 1e-10."""
import numpy as np
import pytest

from helpers import rel_err

pytestmark = pytest.mark.gpu

# (N, intervals, integration, M, density, solver): sizes just past where the
# operator form starts, a last tile of 64 targets that is nearly empty or
# nearly full, scenes whose near pairs outgrow the first store (0.3 and 5 fibers
# per unit volume: 400 and almost all of the sources), and scenes with few.
CASES = [(5, 8, "numerical", 961, 0.03, "gmres"), (5, 8, "analytical", 1023, 0.1, "bicgstab"),
         (5, 16, "numerical", 1000, 0.3, "gmres"), (5, 8, "analytical", 950, 5.0, "gmres"),
         (4, 4, "analytical", 1217, 0.002, "gmres"), (3, 8, "numerical", 1601, 0.05, "gmres"),
         (6, 8, "numerical", 780, 0.05, "bicgstab"), (7, 4, "analytical", 705, 0.03, "gmres"),
         (8, 8, "numerical", 600, 0.05, "gmres")]


def _run(fmt, case, **kw):
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    N, nqi, integration, M, density, solver = case
    pos, ori = cube(M, (M / density) ** (1.0 / 3.0), min_dist=0.4 if density < 1 else 0.1, seed=M)
    params = Parameters(NUMBER_OF_FIBERS=M, NUMBER_OF_TERMS_IN_FORCE_EXPANSION=N, NUMBER_OF_QUADRATURE_INTERVALS=nqi,
                        GMRES_RESTART=30, GMRES_TOLERANCE=1e-10, BICGSTAB_TOLERANCE=1e-10)
    out = {"scene": (pos, ori)}
    with Simulation(params, pos, ori, solver=solver, integration=integration, matrix_format=fmt, **kw) as sim:
        assert sim.step(0) == 0
        out["bytes"] = sim.device_bytes()
        _, out["b"], out["x"] = sim.system()
        assert sim.step(1) == 0
        out["pos"], out["ori"] = sim.state()
        out["v"], out["w"] = sim.velocities()
    return out


@pytest.mark.parametrize("case", CASES)
def test_operator_matches_the_oracle_and_the_stored_form(case):
    from oracle.pyoracle import Oracle, make_params

    a, b = _run("auto", case), _run("theta", case)
    if case[4] < 1:
        assert a["bytes"] < b["bytes"]  # the forms are two
    N, nqi, integration, M = case[:4]
    i0 = M // 3
    rows = slice(3 * N * i0, 3 * N * (i0 + 6))
    A, rhs = Oracle(64).assemble_rows(make_params(M, N=N, nqi=nqi), *a["scene"], i0, i0 + 6,
                                      integration == "analytical")
    residual = np.abs(rhs - A @ a["x"]).max() / np.abs(rhs).max()
    print(f"{case}: b {rel_err(a['b'][rows], rhs):.1e}, residual {residual:.1e}", flush=True)
    assert rel_err(a["b"][rows], rhs) < 4e-6 and residual < 4e-6
    for key in ("pos", "ori", "v", "w"):
        e = rel_err(a[key], b[key])
        print(f"{case}: {key} {e:.1e}", flush=True)
        assert e < 1e-6 if case[4] < 1 else e < 1e-4  # fibers 0.1 apart: condition number ~100 times larger


def test_separate_residual_and_pairwise_velocities():
    """The options that leave parts of the operator out give the same steps."""
    case = CASES[0]
    a = _run("auto", case)
    for kw in ({"separate_residual": True}, {"velocity_operator": "pairwise"}, {"confirm_residual": True},
               {"initial_guess": "extrapolated"}):
        b = _run("auto", case, **kw)
        for key in ("x", "pos", "ori", "v", "w"):
            assert rel_err(b[key], a[key]) < 1e-6, (kw, key)


def test_dumped_matrix_is_the_systems():
    """rf_get_system forms the dense matrix from the state: it matches the stored
    form's, and is refused once the state it belongs to is overwritten."""
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    M = 930
    pos, ori = cube(M, 30.0, min_dist=0.4, seed=1)
    params = Parameters(NUMBER_OF_FIBERS=M)
    A = {}
    for fmt in ("auto", "theta"):
        with Simulation(params, pos, ori, integration="analytical", matrix_format=fmt) as sim:
            sim.assemble_system()
            A[fmt], _, _ = sim.system(with_matrix=True)
            sim.step(0)
            again, _, _ = sim.system(with_matrix=True)
            assert np.array_equal(again, A[fmt])
            sim.step(1)
            sim.set_state(pos, ori)
            sim.assemble_system()
            sim.set_state(ori, pos)
            with pytest.raises(Exception):
                sim.system(with_matrix=True)
    assert rel_err(A["auto"], A["theta"]) < 2e-6


def test_gmres_ir_on_the_operator():
    """GMRES-IR under "auto" refines with the operator's products: the same steps
    as on the stored form and its FP16 copy, to 1e-6."""
    case = (5, 8, "analytical", 980, 0.05, "gmres-ir")
    a, b = _run("auto", case), _run("theta", case)
    assert a["bytes"] < b["bytes"]
    for key in ("x", "pos", "ori", "v", "w"):
        # x's smallest modes carry b's FP32 rounding, 4e-6 of its largest entry
        assert rel_err(a[key], b[key]) < (4e-6 if key == "x" else 1e-6), key
