"""Batched PCG with the blocks dealt evenly to the threads (512 threads, vectors in LDS) against the lane-per-row
kernel on vectors in global memory, which every size can take."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_batch import TOL, _batch, _beams  # noqa: E402


# sizes up to the largest that fits; with problems of a few rows beside it (threads without a
# block, sweeps without a row), and one past it (back to the lane-per-row kernel, coarse operators eliminated in memory)
@pytest.mark.parametrize("lengths", [[43, 1], [64, 8, 45], [52, 2, 63], [75, 20]])
@pytest.mark.parametrize("rows", [0, 64, 128, 512])
@pytest.mark.parametrize("graph", [True, False])
def test_even_batch_matches_lane_per_row(lengths, rows, graph):
    meshes, fixed, mu, lam = _beams(3, lengths)
    out = []
    for lds in (1, 1, 0):
        b = _batch(meshes, fixed, mu, lam, block=512, lanes=1, lds=lds, use_graph=graph, coarse_rows=rows,
                   coarse_period=1)
        kept, infos, _ = b.rollout(2)
        assert all(i["status"] == 0 for step in infos for i in step), infos
        out.append((b, kept, infos))
    (b, kept, infos), (_, again, _), (_, ref, rinfos) = out
    for n in (1, 2):
        assert np.array_equal(kept[n], again[n])
        for p in range(len(lengths)):
            sl = b.problem_slice(p)
            assert np.abs(kept[n][sl] - ref[n][sl]).max() <= TOL * np.abs(ref[n][sl]).max()
            i, r = infos[n - 1][p], rinfos[n - 1][p]
            assert i["newton_iters"] == r["newton_iters"] and i["ls_trials"] == r["ls_trials"]


def test_even_batch_autotunes_and_changes_shape():
    """The assembled order follows the launch shape: set by the tuner, then by hand, on one batch."""
    meshes, fixed, mu, lam = _beams(4, [50, 10])
    b = _batch(meshes, fixed, mu, lam, coarse_rows=64, coarse_period=1)
    b.autotune()
    ref = None
    for shape in [(512, 1, 1), (256, 4, 1), (512, 1, 0), (512, 1, 1)]:
        b._apply_choice(*shape)
        kept, infos, _ = b.rollout(2)
        assert all(i["status"] == 0 for step in infos for i in step), infos
        ref = kept if ref is None else ref
        assert np.abs(kept[2] - ref[2]).max() <= TOL * np.abs(ref[2]).max()
