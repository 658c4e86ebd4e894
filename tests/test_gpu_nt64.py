"""FP64 row-times-row product (k_nt64.hip) through the force bias, at the edges of its
tiles: 16 / 32 / 48 / 64 walkers, 128 Cholesky vectors, K chunks of 16, odd K and
unaligned operands, one and several K ranges.  Every value is compared with a
float64 product on the CPU; a sum of K products is off by at most
(K + ranges) u sum |a b| whatever its order, u = 2^-53, for each side."""

import ctypes

import numpy
import pytest

pytestmark = pytest.mark.gpu

# N, X, na, nb, W
CASES = [
    (2, 1, 1, 1, 1),        # one value of each kind, K below a chunk
    (8, 127, 2, 2, 16),     # one chunk per spin exactly, a column short of a tile
    (9, 129, 3, 2, 17),     # odd K, a row and a column past a tile
    (31, 64, 5, 4, 48),     # odd and even K in the two segments
    (30, 300, 7, 7, 65),    # several K ranges, a row past 64
    (33, 130, 5, 5, 130),   # odd K, three row tiles
    (64, 257, 10, 0, 33),   # one spin
]


def _context(N, X, na, nb, W, offset=0):
    import torch

    from ipie_amd import _lib

    rs = numpy.random.RandomState(N + X + W)
    dev = torch.device("cuda", 0)
    f64, c128 = torch.float64, torch.complex128
    ctx = _lib.Context(N, X, na, nb, W, device=dev)

    def real(*shape):  # `offset` values into its buffer
        n = int(numpy.prod(shape))
        buf = torch.zeros(n + offset, dtype=f64, device=dev)
        buf[offset:] = torch.from_numpy(rs.normal(size=n)).to(dev)
        return buf[offset:].view(*shape)

    ra, rb = real(X, na * N), real(X, nb * N)
    z = lambda *s: torch.zeros(*s, dtype=c128, device=dev)
    ctx.set_static(chol_packed=torch.zeros(N * (N + 1) // 2, X, dtype=f64, device=dev), rchola=ra, rcholb=rb,
                   rH1a=z(na, N), rH1b=z(nb, N), expH1=torch.zeros(2, N, N, dtype=f64, device=dev), mf_shift=z(X),
                   psia=z(N, na), psib=z(N, nb), dt=0.01, ecore=0.0)
    g = [rs.normal(size=(W, n, N)) + 1j * rs.normal(size=(W, n, N)) for n in (na, nb)]
    return ctx, dev, ra.cpu().numpy(), rb.cpu().numpy(), g


def _check(out, ra, rb, g, ranges):
    W = g[0].shape[0]
    want = g[0].reshape(W, -1) @ ra.T + g[1].reshape(W, -1) @ rb.T
    for part in ("real", "imag"):
        size = (numpy.abs(getattr(g[0], part)).reshape(W, -1) @ numpy.abs(ra).T
                + numpy.abs(getattr(g[1], part)).reshape(W, -1) @ numpy.abs(rb).T)
        bound = 2 * (ra.shape[1] + rb.shape[1] + ranges) * 2.0**-53 * size
        assert (numpy.abs(getattr(out, part) - getattr(want, part)) <= bound).all()


@pytest.mark.parametrize("offset", [0, 1])  # rows of B on and off 16 bytes
@pytest.mark.parametrize("case", CASES)
def test_product_at_tile_edges(case, offset):
    import torch

    N, X, na, nb, W = case
    print(f"[case] nt64 N={N} X={X} na={na} nb={nb} W={W} offset={offset}", flush=True)
    ctx, dev, ra, rb, g = _context(N, X, na, nb, W, offset)
    ga, gb = (torch.from_numpy(x).to(dev) for x in g)
    default, lo, hi = ctx.tune_get("fb_split")
    for split in sorted({default, lo, hi}):
        ctx.tune_set("fb_split", split)
        out = torch.empty(W, X, dtype=torch.complex128, device=dev)
        ctx.force_bias(ga, gb, out)
        _check(out.cpu().numpy(), ra, rb, g, split)


def test_product_with_rows_off_sixteen_bytes():
    """A's rows 8 bytes off (a caller of the C entry point)."""
    import torch

    N, X, na, nb, W = 9, 70, 3, 2, 40
    print("[case] nt64 A rows 8 bytes off", flush=True)
    ctx, dev, ra, rb, g = _context(N, X, na, nb, W)
    bufs = []
    for x in g:
        b = torch.zeros(2 * x.size + 1, dtype=torch.float64, device=dev)
        b[1:] = torch.from_numpy(x.view(numpy.float64).ravel()).to(dev)
        bufs.append(b)
    out = torch.empty(W, X, dtype=torch.complex128, device=dev)
    ctx._call("afqmc_force_bias", W, ctypes.c_void_p(bufs[0].data_ptr() + 8),
              ctypes.c_void_p(bufs[1].data_ptr() + 8), ctypes.c_void_p(out.data_ptr()))
    _check(out.cpu().numpy(), ra, rb, g, ctx.tune_get("fb_split")[0])


# N, X, na, nb, W (X > N: the exchange as a quadratic form)
QUAD_CASES = [
    (4, 5, 2, 1, 1),        # less than a column tile
    (16, 20, 8, 8, 17),     # one column tile exactly
    (43, 50, 3, 3, 40),     # a column past a tile, odd n N
    (33, 40, 31, 0, 130),   # eight tiles, the last one short, one spin
    (60, 80, 20, 19, 70),   # several units per tile
]


@pytest.mark.parametrize("case", QUAD_CASES)
def test_quadratic_form_at_tile_edges(case):
    """Coulomb minus exchange of random walkers.  The sums over x, k and c and the
    products of complex numbers are off by at most 4 (X + 2 n N) u of the same sums
    of absolute values, on each side."""
    import torch

    N, X, na, nb, W = case
    print(f"[case] nt64 quadratic form N={N} X={X} na={na} nb={nb} W={W}", flush=True)
    ctx, dev, ra, rb, g = _context(N, X, na, nb, W)
    assert ctx.exchange_form() == "quad"
    ga, gb = (torch.from_numpy(x).to(dev) for x in g)
    out = torch.empty(W, 3, dtype=torch.complex128, device=dev)
    ctx.local_energy(ga, gb, out)
    got = out.cpu().numpy()[:, 2]

    def sums(mag):
        coul, exx = 0.0, 0.0
        for r, x in ((ra, g[0]), (rb, g[1])):
            n = x.shape[1]
            if n == 0:
                continue
            l, y = mag(r.reshape(X, n, N)), mag(x)
            t = numpy.einsum("xim,wjm->wxij", l, y)
            coul = coul + numpy.einsum("wxii->wx", t)
            exx = exx + numpy.einsum("wxij,wxji->w", t, t)
        return 0.5 * (coul * coul).sum(axis=1), 0.5 * exx

    coul, exx = sums(lambda v: v)
    ca, ea = sums(numpy.abs)
    bound = 2 * 4 * (X + 2 * max(na, nb) * N) * 2.0**-53 * (ca + ea)
    assert (numpy.abs(got - (coul - exx)) <= bound).all()
