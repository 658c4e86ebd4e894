"""Green's function and overlap at the edges of their tiles: 1 to 64 occupied orbitals,
spins of different numbers (their eliminations run side by side), basis sizes around
the 16-column tiles, real and complex trials.  Against numpy: with kappa the condition
number of the overlap matrix, the inverse and the determinant are off by at most a
modest multiple of n kappa u."""

import numpy
import pytest

from tests.test_gpu_walker_products import _context

pytestmark = pytest.mark.gpu

# N, na, nb, complex trial, rhf
CASES = [
    (1, 1, 0, False, False),
    (15, 3, 1, True, False),
    (17, 16, 17, False, False),
    (33, 1, 32, True, False),
    (48, 33, 15, False, False),
    (70, 47, 49, False, False),
    (66, 64, 63, True, False),
    (100, 20, 20, False, True),
    (161, 5, 64, False, False),
]


@pytest.mark.parametrize("case", CASES)
def test_against_numpy(case):
    import torch

    N, na, nb, cplx, rhf = case
    W = 3
    print(f"[case] greens N={N} na={na} nb={nb} complex={cplx} rhf={rhf}", flush=True)
    ctx, dev, _, _, phi, rs = _context(N, na, nb, W, 1, seed=3 * N + na, rhf=rhf)
    psi = [rs.normal(size=(N, n)) + 1j * (rs.normal(size=(N, n)) if cplx else 0.0) for n in (na, nb)]
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    f = lambda *s: torch.zeros(*s, dtype=torch.float64, device=dev)
    ctx.set_static(chol_packed=f(N * (N + 1) // 2, 1), rchola=f(1, na * N), rcholb=f(1, nb * N), rH1a=z(na, N),
                   rH1b=z(nb, N), expH1=f(2, N, N), mf_shift=z(1), psia=t(psi[0] + 0j), psib=t(psi[1] + 0j), dt=0.01,
                   ecore=0.0)
    pa, pb = t(phi[0]), t(phi[1])
    ga, gb, ov, ov2 = z(W, na, N), z(W, nb, N), z(W), z(W)
    shift = rs.normal(size=W)
    ctx.greens_function(pa, pb, ga, gb, ov, t(shift))
    ctx.overlap(pa, pb, ov2, t(shift))
    for w in range(W):
        det, tol_det = numpy.exp(-shift[w]) + 0j, 0.0
        for s, (p, q, g, n) in enumerate(((phi[0], psi[0], ga, na), (phi[1], psi[1], gb, nb))):
            if n == 0 or (rhf and s):
                continue
            o = p[w].T @ q.conj()
            sv = numpy.linalg.svd(o, compute_uv=False)
            tol = 100 * n * 2.0**-53 * sv[0] / sv[-1]
            tol_det += (2 if rhf else 1) * tol
            sign, logdet = numpy.linalg.slogdet(o)
            det *= (sign * numpy.exp(logdet)) ** (2 if rhf else 1)
            ref = numpy.linalg.inv(o) @ p[w].T
            assert numpy.abs(g[w].cpu().numpy() - ref).max() <= tol * numpy.abs(ref).max(), (w, s)
        for x in (ov, ov2):
            assert abs(complex(x[w]) / det - 1.0) <= tol_det, (w, complex(x[w]), det)
