"""The resident block-Jacobi PCG (one launch per solve, matrix on chip) against the launch-per-phase
form of the same solver (chosen by giving a chunk length) on the same steps: the two solve each Newton
system to rtol 1e-8 from the same arithmetic in another order of sums, so positions agree to 1e-10
relative per step (the Newton stop at 1e-6 of the start gradient leaves errors of that order times the
second-order convergence) and PCG counts to 3% plus a few iterations. Sizes: one workgroup, a few, odd
boxes, slender ones, rows of every workgroup at the thread count's edge, blocks spilling from registers
to LDS and to the streamed tier, and the default cut of an unnumbered mesh, whose halos are long."""

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

CASES = [((1, 1, 1), "fp64", "snh", True), ((1, 1, 1), "mixed", "snh", True), ((3, 2, 4), "fp64", "arap", True),
         ((7, 7, 7), "mixed", "arap", True), ((9, 5, 11), "fp64", "snh", False), ((16, 16, 16), "fp64", "snh", True),
         ((4, 40, 4), "mixed", "snh", True), ((31, 17, 23), "mixed", "snh", False), ((23, 29, 31), "fp64", "arap", True),
         ((49, 48, 47), "fp64", "snh", True), ((49, 48, 47), "mixed", "arap", True), ((40, 36, 38), "fp64", "snh", False)]


def _box(n, seed):
    from simkit_amd.mesh import jitter, tetrahedralized_grid
    cell = 1.0 / max(n)
    X, T = tetrahedralized_grid(n[0] + 1, n[1] + 1, n[2] + 1, *[k * cell for k in n])
    X = X - X.min(axis=0)
    fixed = np.where(X[:, 1] < 0.5 * cell)[0]
    return jitter(X, cell, 0.1, seed, keep=fixed), T, fixed


@pytest.mark.parametrize("n,precision,material,renumber", CASES)
def test_resident_solve_matches_the_launches(n, precision, material, renumber):
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    X, T, fixed = _box(n, 3)
    mu, lam = ympr_to_lame(1e6, 0.45)
    out = []
    for chunk in (0, 8):  # 8: the launches
        sim = BackwardEulerSim(X, T, mu, lam, rho=1000.0, material=material, fixed_vertices=fixed, gravity=-9.8,
                               precision=precision, renumber=renumber, pcg_chunk=chunk)
        kept, infos = sim.rollout(2)
        assert all(i["status"] == 0 for i in infos), infos
        out.append((kept, infos))
    (k0, i0), (k1, i1) = out
    for s in (1, 2):
        err = np.abs(k0[s] - k1[s]).max() / np.abs(k1[s]).max()
        assert err < 1e-10, (s, err)
        a, b = i0[s - 1], i1[s - 1]
        assert a["newton_iters"] == b["newton_iters"]
        assert abs(a["pcg_iters"] - b["pcg_iters"]) <= 0.03 * b["pcg_iters"] + 4, (a, b)


def test_resident_solve_is_bitwise_deterministic_and_leaves_no_state():
    """Two steps from the same state on one simulator, and on a fresh one, give the same bits."""
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    X, T, fixed = _box((13, 11, 12), 4)
    mu, lam = ympr_to_lame(1e6, 0.45)
    for precision in ("fp64", "mixed"):
        a, b = (BackwardEulerSim(X, T, mu, lam, fixed_vertices=fixed, gravity=-9.8, precision=precision)
                for _ in range(2))
        x = a.X_dev.clone()
        first, _ = a.step(x, x)
        again, _ = a.step(x, x)
        fresh, _ = b.step(x, x)
        assert np.array_equal(first.cpu().numpy(), again.cpu().numpy())
        assert np.array_equal(first.cpu().numpy(), fresh.cpu().numpy())


def test_iteration_limit_and_breakdown_reach_the_caller():
    """The resident solve reports what the launches report: an iteration limit is used as a direction
    (as many iterations as allowed), an indefinite system is a breakdown."""
    from simkit_amd import _lib
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    X, T, fixed = _box((6, 6, 6), 5)
    mu, lam = ympr_to_lame(1e6, 0.45)
    for precision in ("fp64", "mixed"):
        got = []
        for chunk in (0, 8):
            sim = BackwardEulerSim(X, T, mu, lam, fixed_vertices=fixed, gravity=-9.8, precision=precision,
                                   pcg_max_iter=5, newton_max_iter=2, pcg_chunk=chunk)
            x1, info = sim.step(sim.X_dev, sim.X_dev)
            got.append((info["status"], info["pcg_iters"], x1.cpu().numpy()))
        assert got[0][:2] == got[1][:2] and got[0][1] == 10
        assert np.abs(got[0][2] - got[1][2]).max() < (1e-12 if precision == "fp64" else 1e-6)
        squeezed = X * np.array([1.0, 0.3, 1.0])
        sim = BackwardEulerSim(X, T, mu, lam, h=1.0, fixed_vertices=fixed, precision=precision, psd=False)
        xc = sim.X_dev.clone()
        xc.copy_(xc.new_tensor(squeezed.reshape(-1)))
        _, info = sim.step(xc, xc)
        assert info["status"] == _lib.SK_ERR_PCG_BREAKDOWN
