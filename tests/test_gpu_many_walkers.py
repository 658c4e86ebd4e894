"""Green's function and overlap of so many walkers that a workgroup per walker in one grid
dimension would be 2^32 threads, which the runtime refuses: two orbitals, values known
in closed form (products of two numbers per spin, off by a few u)."""

import pytest

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("W", [(1 << 20) + 1, (1 << 23) + 5])
def test_walkers_past_one_grid_dimension(W):
    import torch

    from ipie_amd import _lib

    print(f"[case] walkers W={W}", flush=True)
    dev = torch.device("cuda", 0)
    f = lambda *s: torch.zeros(*s, dtype=torch.float64, device=dev)
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    g = torch.Generator(device=dev)
    g.manual_seed(4)
    ctx = _lib.Context(2, 1, 1, 1, W, device=dev)
    psi = [torch.tensor([[0.6], [0.8]], dtype=torch.complex128, device=dev),
           torch.tensor([[0.8], [-0.6]], dtype=torch.complex128, device=dev)]
    ctx.set_static(chol_packed=f(3, 1), rchola=f(1, 2), rcholb=f(1, 2), rH1a=z(1, 2), rH1b=z(1, 2), expH1=f(2, 2, 2),
                   mf_shift=z(1), psia=psi[0], psib=psi[1], dt=0.01, ecore=0.0)
    phi = [torch.view_as_complex(1.0 + torch.rand(W, 2, 1, 2, dtype=torch.float64, device=dev, generator=g)) + 2.0
           for _ in range(2)]
    o = [(p[:, 0, 0] * q[0, 0] + p[:, 1, 0] * q[1, 0]) for p, q in zip(phi, psi)]
    ga, gb, ov, ov2 = z(W, 1, 2), z(W, 1, 2), z(W), z(W)
    ctx.overlap(*phi, ov)
    ctx.greens_function(*phi, ga, gb, ov2)
    # |o_b| may be a tenth of its two products' sizes: 10 x a few roundings each
    for x in (ov, ov2):
        assert float((x / (o[0] * o[1]) - 1.0).abs().max()) < 1e-13
    for got, p, q in ((ga, phi[0], o[0]), (gb, phi[1], o[1])):
        assert float((got[:, 0] / (p[:, :, 0] / q[:, None]) - 1.0).abs().max()) < 1e-13
