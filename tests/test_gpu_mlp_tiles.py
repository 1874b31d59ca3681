"""The BF16 products and column sums of the MLP at the edges of their tiles."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from oracle import mlp as omlp  # noqa: E402
from test_gpu_mlp import _bf16_bits, _rel  # noqa: E402


@pytest.mark.parametrize("m,n,k", [(16, 16, 16), (48, 80, 64), (32, 96, 80), (176, 64, 208), (1040, 1008, 48),
                                   (1024, 1040, 144)])
@pytest.mark.parametrize("a_t,b_t", [(False, False), (True, False), (False, True)])
@pytest.mark.parametrize("pad", [0, 8, 3])  # 16-byte staging along either dimension, or element by element
def test_gemm_tiles(m, n, k, a_t, b_t, pad):
    from simkit_amd import _lib
    from simkit_amd._device import ptr, stream
    rng = np.random.default_rng(m + n + k)
    A, B = omlp.to_bf16(rng.standard_normal((m, k))), omlp.to_bf16(rng.standard_normal((k, n)))
    store = lambda X, t: _bf16_bits(np.pad(X.T if t else X, ((0, 0), (0, pad))))
    strides = lambda X, t: (1, X.shape[0] + pad) if t else (X.shape[1] + pad, 1)
    Ad, Bd = store(A, a_t), store(B, b_t)
    C = torch.full((m, n), np.nan, dtype=torch.float32, device="cuda")
    _lib.call("sk_gemm_bf16", m, n, k, ptr(Ad), *strides(A, a_t), ptr(Bd), *strides(B, b_t), ptr(C), n, stream())
    # exact products, FP32 sums of k terms: k roundings of at most 2^-23 of the sum of magnitudes
    A, B = np.asarray(A, np.float64), np.asarray(B, np.float64)
    assert (np.abs(C.cpu().numpy() - A @ B) <= k * 2.0 ** -23 * (np.abs(A) @ np.abs(B))).all()


@pytest.mark.parametrize("dims,batch", [((5, 33, 7), 1), ((16, 31, 65, 3), 9), ((70, 64, 32, 40), 257)])
def test_gradient_tiles(dims, batch):
    """Column sums and the GELU'-scaled product over odd widths and batches. FP32 sums in another order can move a
    value over a BF16 rounding boundary: one unit, 2^-8 of the value, in the worst case of every value."""
    from simkit_amd.mlp import MLP
    rng = np.random.default_rng(batch)
    net = MLP(dims, max_batch=batch, seed=1)
    X, T = rng.standard_normal((batch, dims[0])), rng.standard_normal((batch, dims[-1]))
    X, T = X.astype(np.float32), T.astype(np.float32)
    net.backward(torch.from_numpy(X).cuda(), torch.from_numpy(T).cuda())
    _, go = omlp.loss_and_grad(omlp.unflatten(net.get_params(), dims), X, T)
    assert _rel(net.get_grad(), omlp.flatten(go)) < 2.0 ** -8
