"""QR re-orthogonalisation at the edges of its 16-column blocks, with walkers that
pass the condition bound and walkers that go to the shifted three-pass kernel in the
same call (and spins that differ in it)."""

import numpy
import pytest

from tests.test_gpu_walker_products import _context

pytestmark = pytest.mark.gpu

# N, na, nb
CASES = [(1, 1, 0), (15, 15, 1), (16, 16, 0), (18, 17, 16), (40, 32, 31), (70, 33, 1), (101, 48, 47), (66, 49, 48)]


@pytest.mark.parametrize("case", CASES)
def test_blocks_and_mixed_condition(case):
    import torch

    N, na, nb = case
    W = 6
    print(f"[case] reortho N={N} na={na} nb={nb} W={W}", flush=True)
    rs = numpy.random.RandomState(100 + N)
    ctx, dev = _context(N, na, nb, W, 6, seed=N)[:2]
    phi = []
    for s, n in enumerate((na, nb)):
        x = rs.normal(size=(W, N, n)) + 1j * rs.normal(size=(W, N, n))
        for w in (1 + s, 4):  # walkers 1 and 2 ill conditioned in one spin, 4 in both
            if n > 1:
                u, _, v = numpy.linalg.svd(x[w], full_matrices=False)
                x[w] = (u * numpy.logspace(0.0, -6.0, n)) @ v
        phi.append(x)
    ovlp = rs.normal(size=W) + 1j * rs.normal(size=W)
    t = lambda a: torch.from_numpy(a.copy()).to(dev)
    pa, pb, ov = t(phi[0]), t(phi[1]), t(ovlp)
    det, logdet, shift = (torch.zeros(W, dtype=torch.float64, device=dev) for _ in range(3))
    ctx.reortho(pa, pb, ov, det, logdet, shift)
    det_ref = numpy.ones(W)
    kappa = numpy.ones(W)
    for x, dev_q in zip(phi, (pa, pb)):
        n = x.shape[2]
        if n == 0:
            continue
        q = dev_q.cpu().numpy()
        for w in range(W):
            # Q and R move by n kappa u times a modest constant
            sv = numpy.linalg.svd(x[w], compute_uv=False)
            k = sv[0] / sv[-1]
            tol = 1e3 * k * 2.0**-53
            ref, r = numpy.linalg.qr(x[w])
            ph = r.diagonal() / numpy.abs(r.diagonal())
            ref = ref * ph
            det_ref[w] *= numpy.abs(r.diagonal()).prod()
            kappa[w] = max(kappa[w], k)
            assert numpy.abs(q[w].conj().T @ q[w] - numpy.eye(n)).max() < 1e-12, (w, n)
            assert numpy.abs(q[w] - ref).max() < tol, (w, n, k)
    tol = 1e3 * kappa * 2.0**-53 * max(na, nb)
    d = det.cpu().numpy()
    assert (numpy.abs(d / det_ref - 1.0) < tol).all(), d / det_ref - 1.0
    assert (numpy.abs(logdet.cpu().numpy() - numpy.log(det_ref)) < tol).all()
    assert (numpy.abs(ov.cpu().numpy() * d / ovlp - 1.0) < 1e-13).all()
