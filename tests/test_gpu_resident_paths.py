"""Which path a solve takes, and the resident PCG's rare ones: every mesh of the two comparison tests runs where it is
meant to (a comparison of the launches with themselves would pass), a run that gives up is solved by launches, exchange
numbers start over, and runs of several simulators share the device."""
import ctypes
import threading

import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

import test_gpu_resident as bj  # noqa: E402
import test_gpu_resident_two as two  # noqa: E402


def _hook(sim, give_up=0, exchanges=0):
    from simkit_amd import _lib
    _lib.call("sk_sim_resident_hook", sim._h, give_up, exchanges)


def _sim(n, precision="fp64", material="snh", per_agg=0, chunk=0, **kw):
    if per_agg:
        return two._sim(n, precision, material, per_agg, chunk, **kw)
    from simkit_amd.sim import BackwardEulerSim
    from simkit_amd.ympr_to_lame import ympr_to_lame
    X, T, fixed = bj._box(n, 3)
    mu, lam = ympr_to_lame(1e6, 0.45)
    return BackwardEulerSim(X, T, mu, lam, rho=1000.0, material=material, fixed_vertices=fixed, gravity=-9.8,
                            precision=precision, pcg_chunk=chunk, **kw)


@pytest.mark.parametrize("n,precision,material,renumber", bj.CASES)
def test_block_jacobi_cases_run_resident(n, precision, material, renumber):
    sim = _sim(n, precision, material, renumber=renumber)
    _, info = sim.step(sim.X_dev, sim.X_dev)
    print(n, sim.solver_info())
    got = sim.solver_info()
    assert got["workgroups"] > 0 and got["gave_up"] == 0
    assert (got["resident_solves"], got["launch_solves"]) == (info["newton_iters"], 0)
    sim = _sim(n, precision, material, chunk=8, renumber=renumber)
    _, info = sim.step(sim.X_dev, sim.X_dev)
    got = sim.solver_info()
    assert got["workgroups"] == 0 and (got["resident_solves"], got["launch_solves"]) == (0, info["newton_iters"])


# FP64 at 49 x 48 x 47 cells: vectors, halo and the coarse space together exceed the LDS
TWO_LAUNCHES = {((49, 48, 47), "fp64", "snh", 216)}


@pytest.mark.parametrize("n,precision,material,per_agg", two.CASES)
def test_two_level_cases_run_where_they_are_meant_to(n, precision, material, per_agg):
    sim = _sim(n, precision, material, per_agg)
    _, info = sim.step(sim.X_dev, sim.X_dev)
    got, k = sim.solver_info(), info["newton_iters"]
    assert got["gave_up"] == 0
    resident = (n, precision, material, per_agg) not in TWO_LAUNCHES
    assert (got["resident_solves"], got["launch_solves"]) == ((k, 0) if resident else (0, k)), got


def test_two_level_fp64_with_streamed_blocks_matches_the_launches():
    """To the bounds of test_gpu_resident_two, at a size with more blocks a thread than its registers hold (8.2 on average
    against 5)."""
    out = []
    for chunk in (0, 4):
        sim = _sim((42, 43, 44), "fp64", "snh", 216, chunk)
        out.append(sim.rollout(2))
        info = sim.solver_info()
        assert (info["resident_solves"] > 0, info["launch_solves"] > 0) == (chunk == 0, chunk != 0), info
    (k0, i0), (k1, i1) = out
    for s in (1, 2):
        assert np.abs(k0[s] - k1[s]).max() / np.abs(k1[s]).max() < 1e-10
        a, b = i0[s - 1], i1[s - 1]
        assert a["newton_iters"] == b["newton_iters"]
        assert abs(a["pcg_iters"] - b["pcg_iters"]) <= 0.03 * b["pcg_iters"] + 4, (a, b)


FORMS = [("fp64", 0), ("mixed", 0), ("fp64", 100), ("mixed", 100)]


@pytest.mark.parametrize("precision,per_agg", FORMS)
def test_a_run_that_gives_up_is_solved_by_launches(precision, per_agg):
    n = (14, 15, 13)
    # in one numbering the very same launches (two-level: the aggregates' vertices in another order, to the bounds of
    # the comparison tests); the chunk length only says how often the host looks
    kw = {"per_agg": per_agg} if per_agg else {"renumber": False}
    tol, slack = (1e-10, 0.03) if per_agg else (1e-12, 0.0)
    sim, ref = _sim(n, precision, **kw), _sim(n, precision, chunk=8, **kw)
    _hook(sim, give_up=1)
    kept, infos = sim.rollout(2)
    want, winfos = ref.rollout(2)
    assert all(i["status"] == 0 for i in infos), infos
    for s in (1, 2):
        a, b = infos[s - 1]["pcg_iters"], winfos[s - 1]["pcg_iters"]
        assert np.abs(kept[s] - want[s]).max() <= tol * np.abs(want[s]).max()
        assert abs(a - b) <= slack * b + (4 if slack else 0)
    got = sim.solver_info()
    assert (got["resident_solves"], got["gave_up"], got["workgroups"]) == (0, 1, 0), got
    assert got["launch_solves"] == sum(i["newton_iters"] for i in infos)


@pytest.mark.parametrize("precision,per_agg", FORMS)
@pytest.mark.parametrize("n", [(1, 1, 3), (5, 3, 8), (13, 12, 14)])
def test_a_solve_run_to_underflow_has_the_launches_status(n, precision, per_agg):
    """With rtol 0 the residual shrinks until its products underflow. Whatever a solve by launches of the same system
    reports for that, in the same numbering, a simulator that runs resident reports too."""
    kw = {"per_agg": per_agg, "pcg_rtol": 0.0, "pcg_max_iter": 4000, "newton_max_iter": 1}
    sim, ref = _sim(n, precision, **kw), _sim(n, precision, **kw)
    _hook(ref, give_up=1)
    x, info = sim.step(sim.X_dev, sim.X_dev)
    y, want = ref.step(ref.X_dev, ref.X_dev)
    assert ref.solver_info()["gave_up"] == 1
    assert info["status"] == want["status"], (info, want)
    if sim.solver_info()["launch_solves"]:
        assert (x - y).abs().max() == 0.0


@pytest.mark.parametrize("precision,per_agg", FORMS)
@pytest.mark.parametrize("start", [0x70000000 - 40, 0x70000000, 65536 - 40, 65535])
def test_exchange_numbers_start_over_and_wrap_their_tags(precision, per_agg, start):
    """Past 0x70000000 the next run starts at 0 again; the two-level words carry the low 16 bits only."""
    n = (11, 12, 10)
    sim, ref = _sim(n, precision, per_agg=per_agg), _sim(n, precision, per_agg=per_agg)
    _hook(sim, exchanges=start)
    kept, infos = sim.rollout(3)
    want, winfos = ref.rollout(3)
    assert all(np.array_equal(kept[s], want[s]) for s in (1, 2, 3))
    assert [i["pcg_iters"] for i in infos] == [i["pcg_iters"] for i in winfos]
    got, total = sim.solver_info(), ref.solver_info()["exchanges"]
    assert got["launch_solves"] == got["gave_up"] == 0
    assert got["exchanges"] < total if start > 65536 else got["exchanges"] == start + total


def _hip():
    """The HIP runtime that torch and the library have loaded."""
    path = next(line.split()[-1] for line in open("/proc/self/maps") if "libamdhip64.so" in line)
    return ctypes.CDLL(path)


def test_a_stream_with_a_cu_mask_takes_the_launches():
    """Half of the CUs: where its workgroups could run on each XCD is not known, so they must not wait for each other."""
    hip, stream = _hip(), ctypes.c_void_p()
    sim, ref = _sim((9, 8, 10), renumber=False), _sim((9, 8, 10), chunk=8, renumber=False)
    torch.cuda.synchronize()
    mask = (ctypes.c_uint32 * 8)(*[0xFFFFFFFF] * 4 + [0] * 4)
    assert hip.hipExtStreamCreateWithCUMask(ctypes.byref(stream), 8, mask) == 0
    try:
        with torch.cuda.stream(torch.cuda.ExternalStream(stream.value)):
            x1, info = sim.step(sim.X_dev, sim.X_dev)
            torch.cuda.current_stream().synchronize()
        want, _ = ref.step(ref.X_dev, ref.X_dev)
        got = sim.solver_info()
        assert (got["resident_solves"], got["launch_solves"], got["gave_up"]) == (0, info["newton_iters"], 0), got
        assert (x1 - want).abs().max() <= 1e-12 * want.abs().max()
        _, info = sim.step(sim.X_dev, sim.X_dev)  # and on an ordinary stream again resident
        assert sim.solver_info()["resident_solves"] == info["newton_iters"]
    finally:
        assert hip.hipStreamDestroy(stream) == 0


def test_runs_of_several_threads_share_the_device():
    """Simulators stepped by threads of their own on streams of their own: cuts that fit the chip together and cuts that
    need all of it, with workgroup counts that are no multiple of the eight XCDs among them. Nobody gives up, and every
    trajectory is the one its simulator has alone."""
    specs = [((23, 29, 31), "mixed", 216), ((13, 11, 12), "fp64", 100), ((24, 25, 23), "fp64", 0),
             ((4, 40, 4), "fp64", 100), ((9, 5, 11), "mixed", 60)]
    sims = [_sim(n, p, per_agg=a) for n, p, a in specs]
    want = [_sim(n, p, per_agg=a).rollout(4)[0] for n, p, a in specs]
    torch.cuda.synchronize()
    kept, errors = [None] * len(sims), []

    def run(k):
        try:
            stream = torch.cuda.Stream()
            with torch.cuda.stream(stream):
                kept[k] = sims[k].rollout(4)[0]
                stream.synchronize()
        except Exception as e:  # noqa: BLE001 (reported by the main thread)
            errors.append((k, e))

    threads = [threading.Thread(target=run, args=(k,)) for k in range(len(sims))]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not errors, errors
    for sim, got, ref in zip(sims, kept, want):
        info = sim.solver_info()
        assert info["gave_up"] == info["launch_solves"] == 0, info
        assert all(np.array_equal(got[s], ref[s]) for s in range(1, 5))


@pytest.mark.parametrize("precision,per_agg", [("fp64", 0), ("mixed", 0)])
def test_the_first_step_allocates_nothing(precision, per_agg):
    """A numbered simulator has its plan and buffers when it is built: a first step that allocates would wait for
    whatever else runs on the device. (Two-level, the first step still forms the coarse operator.)"""
    warm = _sim((40, 38, 39), precision, per_agg=per_agg)
    warm.step(warm.X_dev, warm.X_dev)  # kernels loaded
    sim = _sim((40, 39, 38), precision, per_agg=per_agg)
    x, out = sim.X_dev, torch.empty_like(sim.X_dev)
    torch.cuda.synchronize()
    free = torch.cuda.mem_get_info()[0]
    sim.step(x, x, out=out)
    torch.cuda.synchronize()
    assert torch.cuda.mem_get_info()[0] == free
    assert sim.solver_info()["launch_solves"] == 0 < sim.solver_info()["resident_solves"]
