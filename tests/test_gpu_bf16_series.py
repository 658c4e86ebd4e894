"""Split-BF16 Taylor series at its edges: atoms of 16, K chunks of 32, groups of 32 columns
with a full or an empty second half, VHS held in LDS (N <= 160), staged (N <= 256) and
a launch per term.  exp(V) phi to `terms` terms against float64 on the CPU, V = i
sqrt(dt) xi_w L for one Cholesky vector.  Each of the first three terms multiplies by V
with operands of 16 significant bits less the lo lo product and FP32 sums: at most 2^-14
of the sum of absolute values; later ones with 8 bits an operand: at most 2^-6."""

import numpy
import pytest

from tests.test_gpu_walker_products import _context

pytestmark = pytest.mark.gpu

# N, na, nb, W, terms
CASES = [
    (2, 1, 0, 1, 6),
    (16, 16, 1, 3, 1),
    (17, 9, 8, 2, 2),
    (33, 16, 16, 3, 6),
    (48, 32, 1, 2, 4),
    (63, 25, 24, 2, 6),
    (159, 10, 7, 2, 6),
    (160, 33, 32, 2, 6),
    (161, 9, 7, 3, 6),
    (192, 40, 40, 2, 3),
    (255, 17, 16, 2, 6),
    (256, 3, 2, 4, 8),
    (257, 9, 8, 2, 6),
]


@pytest.mark.parametrize("case", CASES)
def test_series_at_tile_edges(case):
    import torch

    N, na, nb, W, terms = case
    print(f"[case] split-BF16 series N={N} na={na} nb={nb} W={W} terms={terms}", flush=True)
    ctx, dev, chol, _, phi, rs = _context(N, na, nb, W, terms, seed=N + na, precision="mixed")
    xi = rs.normal(size=(W, 1))
    pa, pb = (torch.from_numpy(p).to(dev) for p in phi)
    ga, gb = (torch.zeros(W, n, N, dtype=torch.complex128, device=dev) for n in (na, nb))
    cmf, cfb = (torch.empty(W, dtype=torch.complex128, device=dev) for _ in range(2))
    ctx.two_body(pa, pb, ga, gb, cmf, cfb, xi=torch.from_numpy(xi).to(dev))
    v = 1j * 0.2 * xi[:, 0, None, None] * chol
    for got, p in ((pa, phi[0]), (pb, phi[1])):
        term, total, aterm, bound = p, p.copy(), numpy.abs(p), numpy.zeros(p.shape)
        for k in range(1, terms + 1):
            term = (v @ term) / k
            aterm = (numpy.abs(v) @ aterm) / k
            total = total + term
            bound = bound + (min(k, 3) * 2.0**-14 + max(k - 3, 0) * 2.0**-6) * aterm
        assert (numpy.abs(got.cpu().numpy() - total) <= bound).all()
