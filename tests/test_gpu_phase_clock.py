"""The per-phase device times (afqmc_profile): the phases of a call follow each other,
so their times add up to no more than an event pair around the call measures, and
to most of it where the kernels take far longer than the launches."""

import pytest

from tests._helpers import Pair, random_walkers, synthetic_arrays

pytestmark = pytest.mark.gpu

# precision, N, na, nb, W, control variate, exp_nmax
CASES = [
    ("fp64", 160, 20, 18, 64, None, 6),
    ("fp64", 160, 50, 50, 32, None, 0),  # no Taylor launch; columns past the fast QR
    ("fp64", 270, 12, 9, 48, None, 6),   # one launch per Taylor term
    ("mixed", 160, 20, 18, 64, None, 6),
    ("mixed", 160, 20, 18, 64, dict(fraction=0.25, warmup=1), 6),
]


@pytest.mark.parametrize("case", CASES, ids=lambda c: f"{c[0]}-{c[1]}-{c[2]}-{'cv' if c[5] else c[6]}")
def test_phases_add_up(case):
    import torch

    precision, N, na, nb, W, sur, nmax = case
    print(f"[case] phases {case}", flush=True)
    h1e, chol, ecore, psi = synthetic_arrays(N, 4 * N, 12.0, na, nb, scale=(12.0 / (N * 12.0)) ** 0.5)
    init = random_walkers(N, na, nb, W, seed=9, amp=0.1, base=psi)
    p = Pair(h1e, chol, psi, (na, nb), W, init=init, precision=precision, surrogate=sur, exp_nmax=nmax)
    ctx = p.prop._engine.ctx
    step = lambda: (p.prop.propagate_walkers(p.walkers, p.ham, p.trial, 0.0), p.walkers.orthogonalise())
    for _ in range(3):  # workspaces and per-set products exist, the warm-up is over
        step()
    ctx.profile(True)
    assert all(ms == 0.0 and n == 0 for ms, n in ctx.profile_read().values())
    start, stop = (torch.cuda.Event(enable_timing=True) for _ in range(2))
    steps = 4
    torch.cuda.synchronize()
    start.record()
    for _ in range(steps):
        step()
    stop.record()
    prof = ctx.profile_read()
    stop.synchronize()
    total, phases = start.elapsed_time(stop), sum(ms for ms, _ in prof.values())
    print(f"total {total:.3f} ms, phases {phases:.3f} ms {prof}", flush=True)
    for ph in ("gf", "force_bias", "fields", "vhs", "taylor", "overlap", "weight", "reortho"):
        assert prof[ph][0] > 0.0 and prof[ph][1] >= steps, ph
    assert all(ms >= 0.0 for ms, _ in prof.values())
    # the clocks' resolution is 10 ns; half of the time may be the host's where
    # kernels outside the phases (copies, the training steps) run between them
    assert phases <= 1.001 * total + 0.01
    assert phases >= 0.5 * total
    ctx.profile(False)
    step()
    ctx.profile(True)
    step()
    ctx.profile(True)  # drops what was stamped before it
    assert all(ms == 0.0 and n == 0 for ms, n in ctx.profile_read().values())
