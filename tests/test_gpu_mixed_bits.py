"""The FP64 values that the mixed step rounds to pairs of BF16 keep their bits.

A value beside a rounding boundary of the pair moves by 2^-17 of itself when its last
bit moves, and a walker by up to 1e-6 with it, so the order of the sums before the
rounding is part of a mixed run's result.  The digests are of the first kernels that
made these values on this GPU (Green's function by LU, QR by the column Cholesky, a
launch per Taylor term summed smallest first); the inputs are numpy's legacy normals,
without a library factorisation."""

import hashlib

import numpy
import pytest

pytestmark = pytest.mark.gpu


def _digest(*tensors):
    h = hashlib.sha256()
    for t in tensors:
        h.update(numpy.ascontiguousarray(t.cpu().numpy()).tobytes())
    return h.hexdigest()[:16]


def _state(N, na, nb, W, rhf):
    import torch

    from ipie_amd import _lib

    X = N + N // 2
    print(f"[case] mixed bits N={N} na={na} nb={nb} W={W} rhf={rhf}", flush=True)
    rs = numpy.random.RandomState(7 * N + W)
    dev = torch.device("cuda", 0)
    t = lambda a: torch.from_numpy(numpy.ascontiguousarray(a)).to(dev)
    cx = lambda *s: rs.normal(size=s) + 1j * rs.normal(size=s)
    scale = 0.3 / numpy.sqrt(N * X)
    psi = numpy.eye(N) + 0.2 / numpy.sqrt(N) * rs.normal(size=(N, N))
    ctx = _lib.Context(N, X, na, nb, W, rhf=rhf, device=dev, precision="mixed")
    ctx.set_static(chol_packed=t(scale * rs.normal(size=(N * (N + 1) // 2, X))),
                   rchola=t(scale * rs.normal(size=(X, na * N))), rcholb=t(scale * rs.normal(size=(X, nb * N))),
                   rH1a=t(cx(na, N)), rH1b=t(cx(nb, N)), expH1=t(numpy.array([numpy.eye(N)] * 2)),
                   mf_shift=t(0.1j * rs.normal(size=X)), psia=t(psi[:, :na] + 0j), psib=t(psi[:, :nb] + 0j), dt=0.01,
                   ecore=0.0)
    phi = [t(psi[None, :, :n] + 0.3 / numpy.sqrt(N) * cx(W, N, n)) for n in (na, nb)]
    z = lambda *s: torch.zeros(*s, dtype=torch.complex128, device=dev)
    return ctx, phi, z


# N, na, nb, W, rhf
CASES = [(24, 5, 4, 10, False), (40, 16, 0, 7, False), (64, 17, 17, 20, True), (101, 10, 9, 33, False),
         (161, 33, 32, 12, False), (255, 25, 48, 9, False), (270, 40, 40, 20, False)]
GREENS = ["26e9584e1888263d", "2536aafa0488bf1b", "dd82cf0016b8290e", "fb9c7ea7d8f8f064",
          "1c60b31bd4c39e85", "19a52dbf8edaafc7", "064982833e9ebe16"]


@pytest.mark.parametrize("case, want", list(zip(CASES, GREENS)))
def test_greens_function(case, want):
    N, na, nb, W, rhf = case
    ctx, phi, z = _state(*case)
    ga, gb, ov = z(W, na, N), z(W, nb, N), z(W)
    ctx.greens_function(*phi, ga, gb, ov)
    assert _digest(ga, gb, ov) == want


QR = ["9d456fa24600893d", "bd9f7ffbf511507a", "347a6b8a9cefe073", "b2ea3f048e36f6f3",
      "c21372017d2d32e3", "b09e3537a776d7b5", "a279fddf69f78a14"]


@pytest.mark.parametrize("case, want", list(zip(CASES, QR)))
def test_reortho(case, want):
    import torch

    N, na, nb, W, rhf = case
    ctx, phi, z = _state(*case)
    det, logdet = (torch.zeros(W, dtype=torch.float64, device=phi[0].device) for _ in range(2))
    ctx.reortho(*phi, z(W), det, logdet)
    assert _digest(*phi, det) == want


STEP = ["ef0c677a9e68a900", "08e2b209ce9f24d2", "aee5d78bfb0f9857", "60706f5073251cc8",
        "0a09d63071a462d0", "cb88c5e06419f963", "3428e7279e1d83f6"]


@pytest.mark.parametrize("case, want", list(zip(CASES, STEP)))
def test_step(case, want):
    N, na, nb, W, rhf = case
    ctx, phi, z = _state(*case)
    g = [p.transpose(1, 2).conj().resolve_conj().contiguous() for p in phi]
    ctx.two_body(*phi, *g, z(W), z(W), seed=3, counter=9)
    ctx.one_body(*phi)
    assert _digest(*phi) == want
