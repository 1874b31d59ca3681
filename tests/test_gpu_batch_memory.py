"""The evenly dealt batched PCG keeps a second copy of the matrix values (36 bytes a block); a batch whose launch shape
does not run it keeps none."""
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from test_gpu_batch import _batch, _beams  # noqa: E402


def test_only_the_dealt_shape_keeps_the_dealt_values():
    meshes, fixed, mu, lam = _beams(5, [40] * 96)
    grown = {}
    for shape in [(256, 1, 0), (512, 1, 1), (256, 1, 0), (512, 1, 1)]:  # the first of each loads its kernels
        b = _batch(meshes, fixed, mu, lam, block=shape[0], lanes=shape[1], lds=shape[2])
        x = b.X_dev
        torch.cuda.synchronize()
        free = torch.cuda.mem_get_info()[0]
        b.step(x, x)
        torch.cuda.synchronize()
        grown[shape] = free - torch.cuda.mem_get_info()[0]
        del b
    copy = 36 * 10 * 25 * 41 * 96  # at least ten blocks a row of 5 x 5 x 41 vertices
    assert grown[512, 1, 1] > 0.9 * copy
    assert grown[256, 1, 0] < 0.1 * copy, grown
