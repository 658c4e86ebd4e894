"""Row products over more than 2^22 values: VHS and force bias of a small basis with many
Cholesky vectors, against float64 on the CPU (a sum of K products is off by at most
(K + ranges) u sum |a b| on each side)."""

import numpy
import pytest

pytestmark = pytest.mark.gpu

U = 2.0**-53


@pytest.mark.parametrize("X", [(1 << 22) - 1, (1 << 22) + 3, (1 << 22) + 1000])
def test_long_rows(X):
    import torch

    from ipie_amd import _lib

    N, W = 2, 3
    print(f"[case] long rows X={X}", flush=True)
    rs = numpy.random.RandomState(3)
    dev = torch.device("cuda", 0)
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    packed, rchol, dt = rs.normal(size=(3, X)), rs.normal(size=(X, N)), 1e-8
    ctx = _lib.Context(N, X, 1, 0, W, exp_nmax=1, device=dev)
    ctx.set_static(chol_packed=t(packed), rchola=t(rchol), rcholb=torch.zeros(X, 0, dtype=torch.float64, device=dev),
                   rH1a=z(1, N), rH1b=z(0, N), expH1=t(numpy.array([numpy.eye(N)] * 2)), mf_shift=z(X), psia=z(N, 1),
                   psib=z(N, 0), dt=dt, ecore=0.0)
    phi = rs.normal(size=(W, N, 1)) + 1j * rs.normal(size=(W, N, 1))
    g = rs.normal(size=(W, 1, N)) + 1j * rs.normal(size=(W, 1, N))
    xi = rs.normal(size=(W, X))
    pa, vb = t(phi), z(W, X)
    ctx.two_body(pa, z(W, N, 0), z(W, 1, N), z(W, 0, N), z(W), z(W), xi=t(xi))
    for w in range(W):
        v = numpy.empty((N, N))
        size = numpy.empty((N, N))
        for p, (i, j) in enumerate(((0, 0), (0, 1), (1, 1))):
            v[i, j] = v[j, i] = packed[p] @ xi[w]
            size[i, j] = size[j, i] = numpy.abs(packed[p]) @ numpy.abs(xi[w])
        want = phi[w] + 1j * numpy.sqrt(dt) * v @ phi[w]
        bound = 2 * (X + 8) * U * (numpy.abs(phi[w]) + numpy.sqrt(dt) * size @ numpy.abs(phi[w])) * 2
        assert (numpy.abs(pa[w].cpu().numpy() - want) <= bound).all()
    ctx.force_bias(t(g), z(W, 0, N), vb)
    want = g[:, 0] @ rchol.T
    assert numpy.abs(vb.cpu().numpy() - want).max() <= 16 * U * (numpy.abs(g[:, 0]) @ numpy.abs(rchol).T).max()
