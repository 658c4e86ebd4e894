"""Operands of the FP64 one body in the caller's memory: expH1 is read in every call, so
that a caller who rewrites it in place is followed, at even and odd N (16- and 4-byte
loads of its rows) and at tile edges, and walkers 8 bytes off (the C entry points take
float64 pairs), loaded 4 bytes a lane.  The product against float64 on the CPU: a
sum of N products is off by at most (N + 2) u sum |a b| on each side."""

import ctypes

import numpy
import pytest

from tests.test_gpu_walker_products import U, _context

pytestmark = pytest.mark.gpu

# N, na, nb, W
CASES = [(1, 1, 1, 2), (2, 2, 1, 3), (15, 3, 0, 5), (16, 4, 4, 4), (17, 5, 4, 13), (31, 8, 7, 40), (32, 9, 9, 33),
         (47, 3, 2, 150), (66, 10, 9, 90), (81, 20, 20, 200), (113, 7, 6, 64)]


def _check(got, exp, phi):
    for s in range(2):
        for part in ("real", "imag"):
            want = numpy.einsum("ik,wkc->wic", exp[s], getattr(phi[s], part))
            size = numpy.einsum("ik,wkc->wic", numpy.abs(exp[s]), numpy.abs(getattr(phi[s], part)))
            bound = 2 * (exp.shape[1] + 2) * U * size
            assert (numpy.abs(getattr(got[s], part) - want) <= bound).all()


@pytest.mark.parametrize("case", CASES)
def test_expH1_rewritten_in_place(case):
    import torch

    N, na, nb, W = case
    print(f"[case] one body N={N} na={na} nb={nb} W={W}", flush=True)
    ctx, dev, _, exp, phi, rs = _context(N, na, nb, W, 6, seed=5 * N + na)
    held = ctx._static_refs[5]  # expH1, which the context borrows
    for values in (exp, rs.normal(size=exp.shape)):
        held.copy_(torch.from_numpy(values))
        out = [torch.from_numpy(p).to(dev) for p in phi]
        ctx.one_body(*out)
        _check([o.cpu().numpy() for o in out], values, phi)


@pytest.mark.parametrize("case", CASES)
def test_walkers_off_sixteen_bytes(case):
    import torch

    N, na, nb, W = case
    print(f"[case] one body, walkers 8 bytes off N={N} na={na} nb={nb} W={W}", flush=True)
    ctx, dev, _, exp, phi, _ = _context(N, na, nb, W, 6, seed=5 * N + na)
    bufs = []
    for p in phi:
        b = torch.zeros(2 * p.size + 1, dtype=torch.float64, device=dev)
        b[1:] = torch.from_numpy(p.view(numpy.float64).ravel()).to(dev)
        bufs.append(b)
    ctx._call("afqmc_one_body", W, *(ctypes.c_void_p(b.data_ptr() + 8) for b in bufs))
    got = [b[1:].cpu().numpy().view(numpy.complex128).reshape(p.shape) for b, p in zip(bufs, phi)]
    assert all(float(b[0]) == 0.0 for b in bufs)
    _check(got, exp, phi)
