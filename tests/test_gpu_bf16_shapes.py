"""Split-BF16 GEMM tile shapes picked by the launch: on either side of the rule's lines
(few and many walkers, short and long K) the force bias, the two-body step and the one
body equal the bits of every shape that can be set, and the quadratic-form exchange,
whose shape is the rule's alone, the FP64 one to the form's accuracy."""

import numpy
import pytest

from tests._helpers import Pair, random_walkers, synthetic_arrays

pytestmark = pytest.mark.gpu

# N, na, nb, W
CASES = [(17, 3, 2, 1), (33, 5, 4, 31), (40, 6, 5, 33), (64, 9, 8, 129), (96, 7, 6, 257), (70, 5, 4, 700)]


@pytest.mark.parametrize("case", CASES)
def test_rule_gives_the_bits_of_every_shape(case):
    import torch

    from ipie_amd.estimators import local_energy_batch

    N, na, nb, W = case
    print(f"[case] shapes N={N} na={na} nb={nb} W={W}", flush=True)
    h1e, chol, ecore, psi = synthetic_arrays(N, 4 * N, 12.0, na, nb, scale=(1.0 / N) ** 0.5)
    init = random_walkers(N, na, nb, W, seed=N, amp=0.1, base=psi)
    p = Pair(h1e, chol, psi, (na, nb), W, init=init, precision="mixed")
    ctx, w = p.walkers._engine.ctx, p.walkers
    ov = p.trial.calc_greens_function(w)
    dev = dict(dtype=torch.complex128, device=w.device)

    def run():
        vb, cmf, cfb = torch.empty(W, 4 * N, **dev), torch.empty(W, **dev), torch.empty(W, **dev)
        ctx.force_bias(w.Ghalfa, w.Ghalfb, vb)
        pa, pb, qa, qb = w.phia.clone(), w.phib.clone(), w.phia.clone(), w.phib.clone()
        ctx.two_body(pa, pb, w.Ghalfa, w.Ghalfb, cmf, cfb, seed=5, counter=3)
        ctx.one_body(qa, qb)
        return [t.cpu().numpy() for t in (vb, pa, pb, cmf, cfb, qa, qb)]

    by_rule = run()
    mixed = local_energy_batch(p.system, p.ham, w, p.trial).cpu().numpy()
    for shape in range(6):
        for knob in ("tile_fb", "tile_vhs", "tile_one_body"):
            ctx.tune_set(knob, shape)
        for a, b in zip(by_rule, run()):
            assert numpy.array_equal(a, b), shape
    q = Pair(h1e, chol, psi, (na, nb), W, init=init)
    assert torch.isfinite(torch.view_as_real(ov)).all()
    q.trial.calc_greens_function(q.walkers)
    exact = local_energy_batch(q.system, q.ham, q.walkers, q.trial).cpu().numpy()
    # three BF16 products of values with 16 significant bits: 2^-15 of the sums' scale
    assert numpy.abs(mixed - exact).max() <= 2.0**-15 * numpy.abs(exact).max()
