"""A launch that is refused opens no phase: the QR of 2^24 walkers is a grid of 2^32
threads, which the runtime does not take, and the phase times stay those of the calls
that ran."""

import pytest

pytestmark = pytest.mark.gpu


def test_refused_launch_leaves_the_phase_times():
    import torch

    from ipie_amd import _lib

    W = 1 << 24
    print(f"[case] refused launch W={W}", flush=True)
    dev = torch.device("cuda", 0)
    f = lambda *s: torch.zeros(*s, dtype=torch.float64, device=dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    ctx = _lib.Context(1, 1, 1, 0, W, device=dev)
    one = torch.ones(1, 1, dtype=torch.complex128, device=dev)
    ctx.set_static(chol_packed=f(1, 1), rchola=f(1, 1), rcholb=f(1, 0), rH1a=z(1, 1), rH1b=z(0, 1), expH1=f(2, 1, 1),
                   mf_shift=z(1), psia=one, psib=z(1, 0), dt=0.01, ecore=0.0)
    phi, det = torch.full((W, 1, 1), 2.0, dtype=torch.complex128, device=dev), f(W)
    ctx.profile(True)
    refused = 0
    for nw in (64, W, 64):
        try:
            ctx._call("afqmc_reortho", nw, _lib.ptr(phi), None, None, _lib.ptr(det), None, None)
        except _lib.AfqmcError as e:
            print(e, flush=True)
            refused += 1
    ms, count = ctx.profile_read()["reortho"]
    print(refused, ms, count, flush=True)
    assert refused == 1 and count == 2
    assert 0.0 < ms < 100.0
    assert float((phi[:64] - 1.0).abs().max()) < 1e-15 and float((phi[64:] - 2.0).abs().max()) == 0.0
