"""The far pairs' node rule (rigidfibers_amd/csrc/rf_device.h, rf_far.hip).

Fibers whose centres lie far_rule's radii apart take their projections
  sum_q w_q P_k(s_q) int P_m(s') K(x_i + s_q t_i - x_j - s' t_j) ds'
(the inner integral by the composite rule, or exact) from NP x NP kernel
values.  On the CPU: the radii are read from the device source, and at each of
them and beyond every projection k, m <= N agrees with the composite one to
1e-8 of the largest G_0 component, also for a thick fiber; fewer nodes miss it.
On the GPU: the assembled system against the FP64 oracle at sizes where the
kernel's blocks of 32 sources are partial, with every mix of near and far.
"""
import os
import re

import numpy as np
import pytest

ROOT = os.path.dirname(os.path.dirname(os.path.abspath(__file__)))


def _radii():
    """{True (4 intervals) or False: (r for np[0], r for np[1]) by N}."""
    with open(os.path.join(ROOT, "rigidfibers_amd", "csrc", "rf_device.h")) as fh:
        src = fh.read()
    out = {}
    for name, key in (("fine", False), ("coarse", True)):
        body = src.split(f"constexpr double {name}[kMaxTerms + 1][2] = {{", 1)[1].split("};", 1)[0] + "}"
        out[key] = [tuple(float(v) for v in p.split(",")) for p in re.findall(r"\{([^{}]*)\}", body)]
        assert len(out[key]) == 9
    return out


def _legendre(n, s):
    return np.stack([np.polynomial.legendre.legval(s, [0] * m + [1]) for m in range(n + 1)])


def _composite(intervals):
    s, w = np.polynomial.legendre.leggauss(3)
    mid = -1.0 + (2.0 * np.arange(intervals) + 1.0) / intervals
    return (mid[:, None] + s / intervals).ravel(), np.tile(w / intervals, intervals)


def _kernel(R, eps):
    r2 = (R * R).sum(-1)
    inv = 1.0 / np.sqrt(r2)
    a = inv + 2.0 * eps ** 2 * inv ** 3
    c = inv ** 3 - 6.0 * eps ** 2 * inv ** 5
    x, y, z = R[..., 0], R[..., 1], R[..., 2]
    return np.stack([a + c * x * x, a + c * y * y, a + c * z * z, c * x * y, c * x * z, c * y * z], -1)


def _lagrange(nodes, s):
    L = np.ones((nodes.size, s.size))
    for p in range(nodes.size):
        for r in range(nodes.size):
            if r != p:
                L[p] *= (s - nodes[r]) / (nodes[p] - nodes[r])
    return L


def _projections(d, ti, tj, left, right, eps):
    (sl, Wl), (sr, Wr) = left, right
    R = d[:, None, None, :] + sl[None, :, None, None] * ti[:, None, None, :] - sr[None, None, :, None] * tj[:, None, None, :]
    return np.einsum("ap,npqc,mq->namc", Wl, _kernel(R, eps), Wr, optimize=True)


def _error(N, intervals, exact, NP, radius, eps=0.01, directions=120):
    rng = np.random.default_rng(100 * N + intervals)

    def unit(n):
        v = rng.normal(size=(n, 3))
        return v / np.linalg.norm(v, axis=1, keepdims=True)

    e, ti, tj = unit(directions), unit(directions), unit(directions)
    ti[:20], tj[10:30] = e[:20], e[10:30]  # fibers along the line of centres
    d = e * (radius * np.where(np.arange(directions) % 3 == 0, 1.0 + rng.random(directions), 1.0))[:, None]
    s, w = _composite(intervals)
    comp = (s, w * _legendre(N, s))
    g, gw = np.polynomial.legendre.leggauss(24)
    full = (g, gw * _legendre(N, g)) if exact else comp
    nodes, _ = np.polynomial.legendre.leggauss(NP)
    ref = _projections(d, ti, tj, comp, full, eps)
    got = _projections(d, ti, tj, *((nodes, W @ _lagrange(nodes, q).T) for q, W in (comp, full)), eps)
    return (np.abs(got - ref).max((1, 2, 3)) / (np.abs(ref[:, 0, 0]).max(1) / 2.0)).max()


@pytest.mark.parametrize("exact", [False, True])
@pytest.mark.parametrize("intervals", [4, 8, 16])
@pytest.mark.parametrize("N", range(1, 9))
def test_rule_at_its_radii(N, intervals, exact):
    for NP, radius in zip((6, 8) if N <= 5 else (8, 10), _radii()[intervals == 4][N]):
        for eps in (0.01, 0.1):
            assert _error(N, intervals, exact, NP, radius, eps) <= 1e-8


def test_fewer_nodes_miss_the_bound():
    far, near = _radii()[False][5]
    assert _error(5, 8, True, 5, far) > 1e-8
    assert _error(5, 8, True, 6, near) > 1e-8


CASES = [(5, 8, True, 449, 0.1, "gmres"), (5, 8, False, 457, 0.1, "gmres"), (5, 8, False, 460, 0.004, "gmres"),
         (1, 8, False, 449, 0.05, "gmres"), (2, 16, False, 480, 0.1, "gmres"), (4, 4, True, 448, 0.02, "gmres"),
         (6, 8, False, 450, 0.05, "gmres"), (7, 4, False, 463, 0.02, "gmres"), (8, 8, True, 448, 0.1, "gmres"),
         (5, 8, True, 451, 0.05, "gmres-ir"), (8, 8, False, 448, 0.05, "gmres-ir")]


@pytest.mark.gpu
@pytest.mark.parametrize("N,nqi,analytical,M,density,solver", CASES)
def test_system_and_steps_against_the_oracle(N, nqi, analytical, M, density, solver):
    """A and b to 2e-6 of their largest entries or three times what the FP32
    oracle is off (near-touching fibers amplify FP32 rounding), and the state
    after a second, warm step (its first residual from the assembly, its
    velocities from the stored operator) to 1e-6: the system's rounding, 4e-8
    of an entry, moves it by 1e-9 a step, a block left out by more than 1e-4."""
    from helpers import rel_err
    from oracle.pyoracle import Oracle, make_params
    from rigidfibers_amd.config import Parameters
    from rigidfibers_amd.scenes import cube
    from rigidfibers_amd.simulation import Simulation

    pos, ori = cube(M, (M / density) ** (1.0 / 3.0), min_dist=0.4, seed=N + M)
    params = Parameters(NUMBER_OF_FIBERS=M, NUMBER_OF_TERMS_IN_FORCE_EXPANSION=N, NUMBER_OF_QUADRATURE_INTERVALS=nqi,
                        GMRES_TOLERANCE=1e-11)
    oracle = Oracle(64)
    p = make_params(M, N=N, nqi=nqi)
    rec = []
    oracle.simulate(p, pos, ori, 2, solver="gmres", analytical=analytical, gmres=(30, 2000, 1e-12), record=rec)
    A, b = oracle.assemble(p, pos, ori, analytical)
    A32, b32 = Oracle(32).assemble(p, pos, ori, analytical)
    with Simulation(params, pos, ori, solver=solver, integration="analytical" if analytical else "numerical") as sim:
        sim.assemble_system()
        Ag, bg, _ = sim.system(with_matrix=True)
        sim.set_state(pos, ori)
        for t in range(2):
            assert sim.step(t) == 0
        pg, og = sim.state()
    assert rel_err(Ag, A) < max(2e-6, 3 * rel_err(A32, A)) and rel_err(bg, b) < max(2e-6, 3 * rel_err(b32, b))
    assert rel_err(pg, rec[1]["pos"]) < 1e-6 and rel_err(og, rec[1]["ori"]) < 1e-6
