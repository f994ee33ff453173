"""The LU's MFMA product by tile (rigidfibers_amd/csrc/rf_gemm.hip): systems whose
panel and trailing products take the tiles of 64, 128 and 256, whole and ragged,
and the capped grid, solved without refinement (a refinement tolerance that the
first solve meets), so that the residual is the factorisation's own.

Bounds: sqrt(n) 2^-24 with a growth of at most 5 for FP32; three roundings of the
packs (2^-9, 2^-12 to nearest, twice for a product of two) for BF16 and FP16."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

BF16, FP16 = 3 * 2 * 2.0 ** -9, 3 * 2 * 2.0 ** -12

# n = 15 M.  A panel has 1024 columns, a trailing update of the 2-byte types
# 3072: 100 -> 476 columns right of the first panel (64); 300 -> 1428 and 3476
# (64, 128); 521 -> 4743 (FP32: 128); 781 -> 8643 (capped 256); 1680 -> 22 128 x
# 3072 (256, a ragged last row of tiles).
CASES = [("direct", 100), ("direct", 300), ("direct", 521), ("mixed-bf16", 100), ("mixed-bf16", 300),
         ("mixed-fp16", 300), ("mixed-bf16", 781), ("mixed-fp16", 781), ("mixed-bf16", 1680), ("mixed-fp16", 1680)]


@pytest.mark.parametrize("solver,M", CASES)
def test_unrefined_solve_by_tile(solver, M):
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    pos, ori = cube(M, (M / 0.03) ** (1.0 / 3.0), min_dist=0.4, seed=M)
    params = Parameters(NUMBER_OF_FIBERS=M, NUMBER_OF_TERMS_IN_FORCE_EXPANSION=5)
    with Simulation(params, pos, ori, solver=solver, integration="numerical", refinement_tolerance=1e9) as sim:
        assert sim.step(0) == 0
        stats, tm = sim.solver_stats(), sim.timings()
    n = 15 * M
    bound = {"direct": 5 * np.sqrt(n) * 2.0 ** -24, "mixed-bf16": BF16, "mixed-fp16": FP16}[solver]
    print(f"{solver} n = {n}: {stats['relative_residual']:.1e} (bound {bound:.1e})", flush=True)
    assert not tm["direct_fallback"] and stats["iterations"] == 0
    assert stats["relative_residual"] < bound
