"""The resident two-level PCG against its launch-per-phase form (chosen by a chunk length), to the bounds of the
block-Jacobi comparison (test_gpu_resident): one aggregate and one workgroup, aggregates cut by workgroups, several
aggregates per workgroup, aggregates with fewer than six motions, blocks spilling from registers to LDS and to the
streamed tier; and sizes that stay with the launches (more aggregates per workgroup than one wave serves)."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_resident import _box  # noqa: E402

CASES = [((1, 1, 1), "fp64", "snh", 216), ((2, 2, 2), "mixed", "snh", 216), ((7, 7, 7), "fp64", "arap", 216),
         ((9, 5, 11), "mixed", "snh", 60), ((4, 40, 4), "fp64", "snh", 100), ((16, 16, 16), "mixed", "arap", 300),
         ((31, 17, 23), "fp64", "snh", 216), ((23, 29, 31), "mixed", "snh", 216), ((49, 48, 47), "fp64", "snh", 216),
         ((49, 48, 47), "mixed", "snh", 400), ((10, 9, 8), "fp64", "snh", 8), ((14, 13, 15), "mixed", "snh", 12)]


def _sim(n, precision, material, per_agg, chunk, **kw):
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    X, T, fixed = _box(n, 3)
    mu, lam = ympr_to_lame(1e6, 0.45)
    return BackwardEulerSim(X, T, mu, lam, rho=1000.0, material=material, fixed_vertices=fixed, gravity=-9.8,
                            precision=precision, preconditioner="two_level", coarse_vertices=per_agg,
                            pcg_chunk=chunk, **kw)


@pytest.mark.parametrize("n,precision,material,per_agg", CASES)
def test_resident_two_level_matches_the_launches(n, precision, material, per_agg):
    out = []
    for chunk in (0, 4):
        kept, infos = _sim(n, precision, material, per_agg, chunk).rollout(2)
        assert all(i["status"] == 0 for i in infos), infos
        out.append((kept, infos))
    (k0, i0), (k1, i1) = out
    for s in (1, 2):
        err = np.abs(k0[s] - k1[s]).max() / np.abs(k1[s]).max()
        assert err < 1e-10, (s, err)
        a, b = i0[s - 1], i1[s - 1]
        assert a["newton_iters"] == b["newton_iters"]
        assert abs(a["pcg_iters"] - b["pcg_iters"]) <= 0.03 * b["pcg_iters"] + 4, (a, b)


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
def test_resident_two_level_is_deterministic_and_keeps_the_iteration_limit(precision):
    a, b = (_sim((13, 11, 12), precision, "snh", 100, 0) for _ in range(2))
    x = a.X_dev.clone()
    first, _ = a.step(x, x)
    again, _ = a.step(x, x)
    fresh, _ = b.step(x, x)
    assert np.array_equal(first.cpu().numpy(), again.cpu().numpy())
    assert np.array_equal(first.cpu().numpy(), fresh.cpu().numpy())
    got = []
    for chunk in (0, 4):
        sim = _sim((6, 6, 6), precision, "snh", 60, chunk, pcg_max_iter=5, newton_max_iter=2)
        x1, info = sim.step(sim.X_dev, sim.X_dev)
        got.append((info["status"], info["pcg_iters"], x1.cpu().numpy()))
    assert got[0][:2] == got[1][:2] and got[0][1] == 10
    assert np.abs(got[0][2] - got[1][2]).max() < (1e-12 if precision == "fp64" else 1e-6)
