"""The rule that picks the split-BF16 tile shapes is the tuning value 0: writing back what
tune_get gives changes no launch, a shape can be left again, and the autotuner times
the rule as the heuristic and keeps it when no shape beats it.  The shape of a launch is
read from its kernel's name."""

import pytest

from tests._helpers import Pair, random_walkers, synthetic_arrays

pytestmark = pytest.mark.gpu

KNOBS = ("tile_fb", "tile_vhs", "tile_one_body")


def _kernels(p):
    """Names of the GEMM kernels of a force bias, a two-body step and a one body."""
    import torch
    from torch.profiler import ProfilerActivity, profile

    ctx, w = p.walkers._engine.ctx, p.walkers
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=w.device)
    vb, cmf, cfb, pa, pb = z(p.W, ctx.dims.nchol), z(p.W), z(p.W), w.phia.clone(), w.phib.clone()
    torch.cuda.synchronize()
    with profile(activities=[ProfilerActivity.CUDA, ProfilerActivity.CPU]) as prof:
        ctx.force_bias(w.Ghalfa, w.Ghalfb, vb)
        ctx.two_body(pa, pb, w.Ghalfa, w.Ghalfb, cmf, cfb, seed=5, counter=3)
        ctx.one_body(pa, pb)
        torch.cuda.synchronize()
    return sorted(e.name for e in prof.events() if "bf16_gemm_kernel" in e.name)


@pytest.mark.parametrize("W", [12, 300])
def test_rule_is_a_value(W):
    from ipie_amd.autotune import Autotuner

    N, na, nb = 96, 9, 8
    print(f"[case] tile rule W={W}", flush=True)
    h1e, chol, _, psi = synthetic_arrays(N, 4 * N, 12.0, na, nb, scale=(1.0 / N) ** 0.5)
    p = Pair(h1e, chol, psi, (na, nb), W, init=random_walkers(N, na, nb, W, seed=2, amp=0.1, base=psi),
             precision="mixed")
    p.trial.calc_greens_function(p.walkers)
    ctx = p.walkers._engine.ctx
    by_rule = _kernels(p)
    assert len(by_rule) > 3
    for knob in KNOBS:
        ctx.tune_set(knob, ctx.tune_get(knob)[0])
    assert _kernels(p) == by_rule
    for knob in KNOBS:
        ctx.tune_set(knob, 4)
    assert _kernels(p) != by_rule
    for knob in KNOBS:
        ctx.tune_set(knob, 0)
    assert _kernels(p) == by_rule
    t = Autotuner(cache_path=None, repeats=1, inner=1, min_gain=1e9, knobs=KNOBS)  # nothing beats the heuristic
    chosen = t.tune_walkers(ctx, p.walkers)
    assert chosen == dict.fromkeys(KNOBS, 0)
    assert _kernels(p) == by_rule
