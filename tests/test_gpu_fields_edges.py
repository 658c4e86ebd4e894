"""Fields of the two-body step where the workgroup's shape changes (up to 126 Cholesky
vectors a wave, few walkers 512 threads, else 256) and where a pair of normals belongs to
two walkers (odd numbers of vectors): the normals are those of draw_normals, cmf and
cfb the float64 sums on the CPU to (X + 64) u of the sums of absolute values; and the
energies' one-body sums at one and several entries a thread."""

import numpy
import pytest

pytestmark = pytest.mark.gpu

U = 2.0**-53
# X, W, N, n
CASES = [(1, 1, 2, 1), (7, 5, 3, 2), (126, 3, 4, 2), (127, 3, 40, 7), (511, 2, 5, 3), (513, 256, 3, 1),
         (513, 257, 3, 1), (601, 600, 33, 4), (2401, 9, 130, 9)]


@pytest.mark.parametrize("case", CASES)
def test_fields_and_energy_sums(case):
    import torch

    from ipie_amd import _lib

    X, W, N, n = case
    print(f"[case] fields X={X} W={W} N={N} n={n}", flush=True)
    rs = numpy.random.RandomState(X + W)
    dev = torch.device("cuda", 0)
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    cx = lambda *s: rs.normal(size=s) + 1j * rs.normal(size=s)
    dt = 0.04
    rchol = rs.normal(size=(2, X, n * N)) / numpy.sqrt(n * N)
    rh1 = [cx(n, N), cx(n, N)]
    mf = 1j * rs.normal(size=X)
    packed = 1e-3 * rs.normal(size=(N * (N + 1) // 2, X))
    ctx = _lib.Context(N, X, n, n, W, device=dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    ctx.set_static(chol_packed=t(packed), rchola=t(rchol[0]), rcholb=t(rchol[1]), rH1a=t(rh1[0]), rH1b=t(rh1[1]),
                   expH1=t(numpy.array([numpy.eye(N)] * 2)), mf_shift=t(mf), psia=z(N, n), psib=z(N, n), dt=dt, ecore=0.5)
    g = [cx(W, n, N), cx(W, n, N)]
    ga, gb = t(g[0]), t(g[1])
    pa, pb, cmf, cfb = t(cx(W, N, n)), t(cx(W, N, n)), z(W), z(W)
    xi_out = torch.empty(W, X, dtype=torch.float64, device=dev)
    vb_out = z(W, X)
    ctx.two_body(pa, pb, ga, gb, cmf, cfb, seed=11, counter=5, xi_out=xi_out, vbias_out=vb_out)
    xi = torch.empty(W * X, dtype=torch.float64, device=dev)
    ctx.draw_normals(xi, 11, 5)
    assert torch.equal(xi_out.flatten(), xi)
    vb, xi = vb_out.cpu().numpy(), xi_out.cpu().numpy()
    xb = -numpy.sqrt(dt) * (1j * vb - mf)
    a = numpy.abs(xb)
    xb = numpy.where(a > 1.0, xb / numpy.where(a > 1.0, a, 1.0), xb)
    for got, terms in ((cmf, -numpy.sqrt(dt) * (xi - xb) * mf), (cfb, xi * xb - 0.5 * xb * xb)):
        bound = (X + 64) * U * numpy.abs(terms).sum(1) * 2
        assert (numpy.abs(got.cpu().numpy() - terms.sum(1)) <= bound).all()
    energy = z(W, 3)
    ctx.local_energy(ga, gb, energy)
    terms = [(g[s] * rh1[s]).reshape(W, -1) for s in range(2)]
    bound = (2 * n * N + 64) * U * (sum(numpy.abs(x).sum(1) for x in terms) + 0.5) * 2
    assert (numpy.abs(energy[:, 1].cpu().numpy() - sum(x.sum(1) for x in terms) - 0.5) <= bound).all()
