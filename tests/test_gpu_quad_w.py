"""W' of the quadratic-form exchange at the edges of its 128-column product tiles, 128- and
160-column output tiles and orbital blocks: the exchange of random Ghalf against
sum_x tr(T_x T_x) in float64 on the CPU.  FP64: (n N + X + 64) u of the sums of absolute
values; mixed: W' and Ghalf in 16 significant bits and FP32 sums, 2^-13 of the largest
walker's sum of absolute values."""

import numpy
import pytest

from ipie_amd import _lib

pytestmark = pytest.mark.gpu

# N, na, nb, X, W
CASES = [(2, 1, 1, 3, 1), (9, 7, 5, 17, 3), (31, 4, 5, 33, 5), (32, 4, 4, 48, 2), (43, 3, 6, 50, 4), (64, 5, 2, 65, 3),
         (75, 11, 3, 90, 2), (128, 2, 3, 131, 3)]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("case", CASES)
def test_exchange_of_random_ghalf(case, precision):
    import torch

    N, na, nb, X, W = case
    print(f"[case] quad W' N={N} na={na} nb={nb} X={X} W={W} {precision}", flush=True)
    rs = numpy.random.RandomState(N + X)
    dev = torch.device("cuda", 0)
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    rchol = [rs.normal(size=(X, n, N)) for n in (na, nb)]
    g = [rs.normal(size=(W, n, N)) + 1j * rs.normal(size=(W, n, N)) for n in (na, nb)]
    ctx = _lib.Context(N, X, na, nb, W, device=dev, precision=precision)
    assert ctx.exchange_form() == "quad"
    ctx.set_static(chol_packed=t(numpy.zeros((N * (N + 1) // 2, X))), rchola=t(rchol[0].reshape(X, -1)),
                   rcholb=t(rchol[1].reshape(X, -1)), rH1a=z(na, N), rH1b=z(nb, N), expH1=t(numpy.zeros((2, N, N))),
                   mf_shift=z(X), psia=z(N, na), psib=z(N, nb), dt=0.01, ecore=0.0)
    energy, vb = z(W, 3), z(W, X)
    ctx.local_energy(t(g[0]), t(g[1]), energy)
    ctx.force_bias(t(g[0]), t(g[1]), vb)
    coul = 0.5 * (vb.cpu().numpy() ** 2).sum(1)
    exx, aexx = numpy.zeros(W, dtype=complex), numpy.zeros(W)
    for r, gg in zip(rchol, g):
        T = numpy.einsum("xim,wjm->wxij", r, gg)
        A = numpy.einsum("xim,wjm->wxij", numpy.abs(r), numpy.abs(gg.real) + numpy.abs(gg.imag))
        exx += numpy.einsum("wxij,wxji->w", T, T)
        aexx += numpy.einsum("wxij,wxji->w", A, A)
    got = 2.0 * (coul - energy[:, 2].cpu().numpy())
    if precision == "fp64":
        bound = (max(na, nb) * N + X + 64) * 2.0**-53 * 4 * (aexx + 2 * numpy.abs(coul))
    else:
        bound = 2.0**-13 * aexx.max()
    assert (numpy.abs(got - exx) <= bound).all(), numpy.abs(got - exx) / bound
