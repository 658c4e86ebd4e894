"""What a last bit before the BF16 split does to a mixed step, on the CPU emulation: a
value beside a rounding boundary of the split moves by one place of its low half, at most
2^-16 of itself, and the walker by that times the size of VHS; a value
elsewhere moves nothing.  So two builds whose FP64 values differ in the last bit agree to
2e-16 but for a walker now and then (tests/test_gpu_mixed_bits.py keeps the bits)."""

import numpy

from tests import _mixed_emu as emu


def _held(x):
    return float(emu.planes_value(numpy.array([x]))[0])


def _boundary(rs):
    """Two neighbouring FP64 values that the split takes to different pairs."""
    a = rs.normal() + 2.0
    b = a + 2.0**-14 * abs(a)
    assert _held(a) != _held(b)
    while numpy.nextafter(a, b) < b:
        m = a + 0.5 * (b - a)
        a, b = (m, b) if _held(m) == _held(a) else (a, m)
    return a, b


def test_one_unit_in_the_last_place():
    rs = numpy.random.RandomState(2)
    N, n = 40, 5
    a = rs.normal(size=(N, N))
    V = 0.35j * (a + a.T) / numpy.abs(numpy.linalg.eigvalsh(a + a.T)).max()
    moved = 0
    for _ in range(20):
        phi = rs.normal(size=(1, N, n)) + 1j * rs.normal(size=(1, N, n))
        x, y = _boundary(rs)
        below, above = phi.copy(), phi.copy()
        below[0, 3, 2], above[0, 3, 2] = x, y
        d_split = abs(_held(y) - _held(x))
        assert d_split <= 2.0**-16 * abs(x)
        moved += d_split >= 2.0**-20 * abs(x)  # (a small low half has a small spacing)
        d = emu.taylor(above, V[None])[0] - emu.taylor(below, V[None])[0]
        d[3, 2] -= above[0, 3, 2] - below[0, 3, 2]
        assert numpy.abs(numpy.delete(d, 2, axis=1)).max() == 0.0  # the other columns keep every bit
        # |V|_2 = 0.35 carries the jump on, and the products' FP32 sums round it
        assert numpy.abs(d).max() <= 0.35 * d_split * 1.5 + 2.0**-20
    assert moved >= 15
    phi = rs.normal(size=(1, N, n)) + 1j * rs.normal(size=(1, N, n))
    other = phi.copy()
    other[0, 3, 2] = numpy.nextafter(phi[0, 3, 2].real, 9.0) + 1j * phi[0, 3, 2].imag
    d = emu.taylor(other, V[None])[0] - emu.taylor(phi, V[None])[0]
    assert numpy.abs(d).max() <= 2.0**-51  # away from a boundary: the value itself, no more
