"""Rounding errors of the one-kernel Green's function (double precision) beside those of
the LU form (mixed precision's FP64 Green's function), both against 80-bit elimination
on the host: Ghalf and overlap, rms over walkers and sizes, are no larger."""

import numpy
import pytest

pytestmark = pytest.mark.gpu

L = numpy.clongdouble


def _product(a, b):
    return numpy.stack([(row[:, None] * b).sum(0) for row in a])


def _inverse(o):
    n = o.shape[0]
    a, det = numpy.concatenate([o, numpy.eye(n, dtype=L)], 1), L(1)
    for k in range(n):
        p = k + int(numpy.argmax(numpy.abs(a[k:, k])))
        if p != k:
            a[[k, p]] = a[[p, k]]
            det = -det
        det *= a[k, k]
        a[k] /= a[k, k]
        f = a[:, k].copy()
        f[k] = 0
        a -= f[:, None] * a[k][None]
    return a[:, n:], det


def test_errors_no_larger_than_lu():
    import torch

    from ipie_amd import _lib

    dev = torch.device("cuda", 0)
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    f = lambda *s: torch.zeros(*s, dtype=torch.float64, device=dev)
    err = {"fp64": ([], []), "mixed": ([], [])}
    for N, na, nb, W in ((60, 6, 5, 12), (120, 17, 12, 10), (200, 40, 38, 8)):
        print(f"[case] Green's function errors N={N} na={na} nb={nb}", flush=True)
        rs = numpy.random.RandomState(N)
        psi = numpy.eye(N) + 0.2 / numpy.sqrt(N) * rs.normal(size=(N, N))
        phi = [psi[None, :, :n] + 0.3 / numpy.sqrt(N) * (rs.normal(size=(W, N, n)) + 1j * rs.normal(size=(W, N, n)))
               for n in (na, nb)]
        got = {}
        for precision in err:
            ctx = _lib.Context(N, N, na, nb, W, device=dev, precision=precision)
            ctx.set_static(chol_packed=f(N * (N + 1) // 2, N), rchola=f(N, na * N), rcholb=f(N, nb * N), rH1a=z(na, N),
                           rH1b=z(nb, N), expH1=f(2, N, N), mf_shift=z(N), psia=t(psi[:, :na] + 0j),
                           psib=t(psi[:, :nb] + 0j), dt=0.01, ecore=0.0)
            ga, gb, ov = z(W, na, N), z(W, nb, N), z(W)
            ctx.greens_function(t(phi[0]), t(phi[1]), ga, gb, ov)
            got[precision] = (ga.cpu().numpy(), gb.cpu().numpy(), ov.cpu().numpy())
        for w in range(W):
            det, ghalf = L(1), []
            for s, n in enumerate((na, nb)):
                p = phi[s][w].astype(L)
                inv, d = _inverse(_product(p.T, psi[:, :n].astype(L)))
                det *= d
                ghalf.append(_product(inv, p.T))
            for precision, (g_err, o_err) in err.items():
                for s in range(2):
                    d = (got[precision][s][w] - ghalf[s]).astype(complex)
                    g_err.append(numpy.linalg.norm(d) / numpy.linalg.norm(ghalf[s].astype(complex)))
                o_err.append(abs(complex(got[precision][2][w] / det - 1)))
    rms = {k: [float(numpy.sqrt(numpy.mean(numpy.square(e)))) for e in v] for k, v in err.items()}
    print(rms, flush=True)
    # 30 walkers: the rms of their overlaps' errors is known to about 1 / sqrt(2 x 30) = 13% on each side
    assert rms["fp64"][0] <= 1.1 * rms["mixed"][0]
    assert rms["fp64"][1] <= 1.3 * rms["mixed"][1]
    assert rms["fp64"][0] < 8 * 2.0**-53 and rms["fp64"][1] < 80 * 2.0**-53
