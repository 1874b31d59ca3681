"""Element staging and the gathers at the edges of their waves and lists: any corner order, any number of tets per
vertex, vertices without a tet, tets that have a vertex twice."""
import numpy as np
import pytest

torch = pytest.importorskip("torch")
pytestmark = pytest.mark.gpu

from conftest import rel_err  # noqa: E402
from oracle import fem  # noqa: E402


@pytest.mark.parametrize("nt,nv", [(1, 4), (1, 9), (63, 20), (64, 64), (65, 300), (257, 40), (1500, 30), (3000, 2500)])
@pytest.mark.parametrize("repeated", [False, True])
@pytest.mark.parametrize("psd", [0, 1])
def test_hessian_and_gradient_of_any_connectivity(nt, nv, repeated, psd):
    from simkit_amd import _lib
    from simkit_amd._device import dev, host
    from simkit_amd._mesh import DeviceMesh
    rng = np.random.default_rng(nt + nv)
    T = np.array([rng.choice(nv, 4, replace=repeated) for _ in range(nt)])
    if repeated:
        T[0, 3] = T[0, 1]
    D = rng.standard_normal((nt, 3, 4))
    x = rng.standard_normal((nv, 3))
    mu, lam, vol = (rng.uniform(0.5, 2.0, nt) for _ in range(3))
    mesh = DeviceMesh(T, dev(D.reshape(-1)), nv)
    args = (_lib.SK_LINEAR, dev(x.reshape(-1)), dev(mu), dev(lam), dev(vol))
    J = fem.deformation_jacobian(D, T, nv)
    ref = fem.hessian_x("linear", x, J, mu[:, None], lam[:, None], vol, bool(psd)).toarray()
    assert rel_err(mesh.to_csr(mesh.hessian(*args, psd)).toarray(), ref) < 1e-10
    gref = fem.gradient_x("linear", x, J, mu[:, None], lam[:, None], vol).reshape(-1)
    assert rel_err(host(mesh.gradient(*args)), gref) < 1e-10
