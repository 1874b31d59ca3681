"""The resident two-level PCG far below the usual tolerances: its restricted residual is updated beside the residual and
must not part from it. Counts and positions as the launches have them, to the bounds of test_gpu_resident_two; a run that
parts ends at the iteration limit with a direction that the line search refuses."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

from test_gpu_resident import _box  # noqa: E402


def _run(n, h, free, rtol, chunk, precision="fp64", inner=1e-2, give_up=False):
    from simkit_amd import _lib
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    import torch
    X, T, fixed = _box(n, 3)
    mu, lam = ympr_to_lame(1e6, 0.45)
    sim = BackwardEulerSim(X, T, mu, lam, rho=1000.0, h=h, fixed_vertices=() if free else fixed, gravity=-9.8,
                           precision=precision, preconditioner="two_level", pcg_rtol=rtol, inner_rtol=inner,
                           pcg_max_iter=4000, newton_max_iter=1, pcg_chunk=chunk)
    if give_up:  # by launches, in the same numbering
        _lib.call("sk_sim_resident_hook", sim._h, 1, 0)
    noise = np.random.default_rng(1).standard_normal(X.size) * 0.01 / max(n)
    x, info = sim.step(sim.X_dev + torch.from_numpy(noise).cuda(), sim.X_dev)
    return x.cpu().numpy(), info, sim.solver_info()


@pytest.mark.parametrize("n", [(3, 8, 13), (16, 16, 16), (24, 24, 24)])
@pytest.mark.parametrize("h,free", [(1 / 60, False), (1.0, False), (1 / 60, True), (1.0, True)])
@pytest.mark.parametrize("rtol", [1e-12, 1e-16, 1e-20])
def test_fp64_solves_below_rounding_converge_like_the_launches(n, h, free, rtol):
    x, info, path = _run(n, h, free, rtol, 0)
    y, ref, _ = _run(n, h, free, rtol, 4)
    assert path["launch_solves"] == 0
    assert info["ls_trials"] == ref["ls_trials"] and info["status"] == ref["status"]
    assert ref["pcg_iters"] < 4000
    assert abs(info["pcg_iters"] - ref["pcg_iters"]) <= 0.03 * ref["pcg_iters"] + 4, (info, ref)
    assert np.abs(x - y).max() <= 1e-10 * np.abs(y).max()


@pytest.mark.parametrize("inner", [1e-3, 1e-4])
def test_mixed_segments_as_deep_as_fp32_goes(inner):
    # against the launches on the same FP32 matrix: in another numbering it is rounded differently
    x, info, path = _run((16, 16, 16), 1.0, False, 1e-10, 0, "mixed", inner)
    y, ref, launches = _run((16, 16, 16), 1.0, False, 1e-10, 0, "mixed", inner, give_up=True)
    assert path["launch_solves"] == 0 == launches["resident_solves"]
    assert info["status"] == ref["status"] and info["refine_steps"] == ref["refine_steps"]
    assert abs(info["pcg_iters"] - ref["pcg_iters"]) <= 0.03 * ref["pcg_iters"] + 4, (info, ref)
    assert np.abs(x - y).max() <= 1e-8 * np.abs(y).max()
