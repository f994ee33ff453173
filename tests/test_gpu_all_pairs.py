"""The theta form's kernels on both sides of far_min_fibers (rigidfibers_amd/csrc/rf_internal.h:
320 fibers with numerical, 448 with exact integrals).  A served batch forms the
suspensions below it with the kernel of every pair, the others, which come first
in its table of targets, with the far and near kernels; each result is bitwise the
one served alone, and follows the single simulation (the same kernels, the product
with the initial guess formed another way) to the solver's tolerance of 1e-10."""
import numpy as np
import pytest

from helpers import ref_config, rel_err

pytestmark = pytest.mark.gpu

SIZES = {"numerical": [40, 321, 17, 320, 319, 64], "analytical": [447, 30, 449, 448, 16]}


def _params(M):
    p = ref_config(validate=False)
    p.NUMBER_OF_FIBERS = M
    p.GMRES_TOLERANCE = 1e-10
    return p


@pytest.mark.parametrize("integration", ["numerical", "analytical"])
def test_served_mix_across_the_line(integration):
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.serve import Server
    from rigidfibers_amd.simulation import Simulation

    steps = 3
    reqs = [(M, *cube(M, (10.0 * M) ** (1 / 3), min_dist=0.4, seed=50 + k)) for k, M in
            enumerate(SIZES[integration])]

    def serve(srv, batch):
        ids = [(srv.submit(pos, ori, steps), M) for M, pos, ori in batch]
        for rid, _ in ids:
            assert srv.wait(rid, timeout=60.0)
        return [srv.collect(rid, M, steps) for rid, M in ids]

    with Server(_params(1), integration=integration, max_active=8) as srv:
        alone = [serve(srv, [r])[0] for r in reqs]
        mixed = serve(srv, reqs)
    for (M, pos, ori), a, b in zip(reqs, alone, mixed):
        assert a["info"]["status"] == 0 and b["info"]["status"] == 0
        assert np.array_equal(a["positions"], b["positions"])
        assert np.array_equal(a["orientations"], b["orientations"])
        with Simulation(_params(M), pos, ori, solver="gmres", integration=integration) as sim:
            for t in range(steps):
                assert sim.step(t) == 0
            p, o = sim.state()
        ep, eo = rel_err(a["positions"], p), rel_err(a["orientations"], o)
        print(f"{integration} M={M}: pos {ep:.1e} ori {eo:.1e}", flush=True)
        assert ep < 1e-8 and eo < 1e-8


@pytest.mark.parametrize("solver,integration,M", [("gmres", "numerical", 319), ("gmres", "analytical", 447),
                                                  ("gmres-ir", "analytical", 33), ("gmres-ir", "numerical", 311),
                                                  ("bicgstab", "analytical", 5)])
def test_first_residual_of_the_assembly(solver, integration, M):
    """The warm steps take their first residual from the assembly (in the sweeps, or
    read back with the FP16 copy); separate_residual forms it with a product."""
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    pos, ori = cube(M, (10.0 * M) ** (1 / 3), min_dist=0.4, seed=M)
    out = []
    for separate in (False, True):
        p = _params(M)
        p.BICGSTAB_TOLERANCE = 1e-10
        with Simulation(p, pos, ori, solver=solver, integration=integration, separate_residual=separate) as sim:
            its = []
            for t in range(3):
                assert sim.step(t) == 0
                its.append(sim.solver_stats()["iterations"])
            out.append((*sim.state(), sim.system()[2], its))
    (p0, o0, x0, i0), (p1, o1, x1, i1) = out
    assert i0 == i1  # a wrong residual would cost the warm steps iterations
    for a, b in ((p0, p1), (o0, o1), (x0, x1)):
        assert rel_err(a, b) < 1e-8
