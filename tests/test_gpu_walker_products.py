"""FP64 one-body product and Taylor series (k_gemm.hip) at the edges of their tiles: row
tiles of 16, K chunks of 16, 8-column blocks, the series in one launch (N <= 128
with V in registers, N <= 256) and a launch per term.  With zero force bias and
mean field the two-body step is exp(V) phi to exp_nmax terms, V = i sqrt(dt) xi_w L for
one Cholesky vector; the float64 sums on the CPU are off by at most (4 N + 8) u per
term of the series of absolute values, on each side."""

import numpy
import pytest

pytestmark = pytest.mark.gpu

U = 2.0**-53
# N, na, nb, W, exp_nmax
CASES = [
    (1, 1, 0, 1, 6),
    (15, 3, 1, 3, 1),       # below one tile, a single term
    (40, 4, 3, 2, 0),       # no terms: the walkers unchanged
    (17, 5, 4, 2, 2),       # one past a tile
    (24, 12, 12, 10, 6),    # columns of three 8-column blocks exactly
    (113, 13, 12, 5, 6),    # eight row tiles, the last with one row
    (128, 9, 0, 3, 6),
    (129, 20, 17, 3, 6),    # past the register-resident form
    (256, 33, 32, 2, 3),
    (257, 41, 40, 2, 6),    # a launch per term, columns past 80
    (330, 9, 8, 3, 3),
]


def _context(N, na, nb, W, terms, seed, rhf=False, precision="fp64"):
    import torch

    from ipie_amd import _lib

    rs = numpy.random.RandomState(seed)
    dev = torch.device("cuda", 0)
    f64, c128 = torch.float64, torch.complex128
    a = rs.normal(size=(N, N))
    chol = (a + a.T) / numpy.sqrt(8.0 * N)
    packed = torch.from_numpy(chol[numpy.triu_indices(N)].reshape(-1, 1).copy()).to(dev)
    exp = rs.normal(size=(2, N, N))
    z = lambda *s: torch.zeros(*s, dtype=c128, device=dev)
    ctx = _lib.Context(N, 1, na, nb, W, exp_nmax=terms, rhf=rhf, device=dev, precision=precision)
    ctx.set_static(chol_packed=packed, rchola=torch.zeros(1, na * N, dtype=f64, device=dev),
                   rcholb=torch.zeros(1, nb * N, dtype=f64, device=dev), rH1a=z(na, N), rH1b=z(nb, N),
                   expH1=torch.from_numpy(exp).to(dev), mf_shift=z(1), psia=z(N, na), psib=z(N, nb), dt=0.04, ecore=0.0)
    phi = [rs.normal(size=(W, N, n)) + 1j * rs.normal(size=(W, N, n)) for n in (na, nb)]
    return ctx, dev, chol, exp, phi, rs


@pytest.mark.parametrize("case", CASES)
def test_series_at_tile_edges(case):
    import torch

    N, na, nb, W, terms = case
    print(f"[case] series N={N} na={na} nb={nb} W={W} terms={terms}", flush=True)
    ctx, dev, chol, _, phi, rs = _context(N, na, nb, W, terms, seed=N + na)
    xi = rs.normal(size=(W, 1))
    pa, pb = (torch.from_numpy(p).to(dev) for p in phi)
    ga, gb = (torch.zeros(W, n, N, dtype=torch.complex128, device=dev) for n in (na, nb))
    cmf, cfb = (torch.empty(W, dtype=torch.complex128, device=dev) for _ in range(2))
    ctx.two_body(pa, pb, ga, gb, cmf, cfb, xi=torch.from_numpy(xi).to(dev))
    v = 1j * 0.2 * xi[:, 0, None, None] * chol
    for got, p in ((pa, phi[0]), (pb, phi[1])):
        term, total, aterm, bound = p, p.copy(), numpy.abs(p), numpy.abs(p)
        for k in range(1, terms + 1):
            term = (v @ term) / k
            aterm = (numpy.abs(v) @ aterm) / k
            total = total + term
            bound = bound + aterm
        assert (numpy.abs(got.cpu().numpy() - total) <= 2 * terms * (4 * N + 8) * U * bound).all()


@pytest.mark.parametrize("case", CASES)
def test_one_body_at_tile_edges(case):
    import torch

    N, na, nb, W, _ = case
    print(f"[case] one body N={N} na={na} nb={nb} W={W}", flush=True)
    ctx, dev, _, exp, phi, _ = _context(N, na, nb, W, 1, seed=N + na)
    pa, pb = (torch.from_numpy(p).to(dev) for p in phi)
    ctx.one_body(pa, pb)
    for got, e, p in ((pa, exp[0], phi[0]), (pb, exp[1], phi[1])):
        for part in ("real", "imag"):
            x = getattr(p, part)
            bound = 2 * (N + 2) * U * (numpy.abs(e) @ numpy.abs(x))
            assert (numpy.abs(getattr(got.cpu().numpy(), part) - e @ x) <= bound).all()
