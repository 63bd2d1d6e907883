"""The LU panel kernel at the edges of its groups of 8 columns, its panels of 32 and its waves of 64 rows:
inverse and log det of random complex matrices against numpy, with rows that force interchanges (graded
magnitudes), a matrix whose columns vanish below the diagonal until late, and odd row strides (the
unaligned path).  The matrices have condition numbers below 1e5: residual of the inverse below
n cond 2^-53 = 1e-9 for n <= 130, log det to 1e-10."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

isle = pytest.importorskip("isle_amd")


@pytest.mark.parametrize("n", [1, 2, 7, 8, 9, 15, 16, 17, 24, 31, 32, 33, 40, 41, 63, 64, 65, 72, 96, 97, 128, 129])
@pytest.mark.parametrize("kind", ["random", "graded", "triangular"])
def test_inverse_and_logdet(n, kind):
    print(f"LU panel n={n} {kind}", flush=True)
    rs = np.random.RandomState(100 + n)
    a = rs.normal(size=(n, n)) + 1j * rs.normal(size=(n, n)) + 2 * np.sqrt(n) * np.eye(n)
    if kind == "graded":  # every pivot comes from below: rows reversed, growing magnitudes
        a = a[::-1] * np.logspace(-1, 1, n)[:, None]
    if kind == "triangular":  # zero columns below the diagonal: pivots stay in place, multipliers 0
        a = np.triu(a)
    inv = isle.invert(a).cpu().numpy()
    assert np.abs(inv @ a - np.eye(n)).max() < 1e-9
    sign, mag = np.linalg.slogdet(a)
    got = isle.logdet(a)
    assert abs(got.real - mag) < 1e-10 * max(1.0, abs(mag))
    assert abs(np.exp(1j * got.imag) - sign) < 1e-10


@pytest.mark.parametrize("n", [160, 255, 288, 321, 480, 511, 512, 513, 545, 600])
def test_strips_and_tall_panels(n):
    """Strips of several row tiles per wave, up to the last panel held in registers (512 rows), one row
    more, and matrices whose first panels are taller and whose later ones are not; scaled rows, so that
    rows are interchanged across panels.  cond < 1e5 (row scaling 10 times the random part's): residual
    below n cond 2^-53 < 1e-8."""
    print(f"LU strips n={n}", flush=True)
    rs = np.random.RandomState(n)
    a = rs.normal(size=(n, n)) + 1j * rs.normal(size=(n, n)) + 2 * np.sqrt(n) * np.eye(n)
    a = a[rs.permutation(n)] * np.exp(rs.uniform(-1, 1, n))[:, None]
    inv = isle.invert(a).cpu().numpy()
    assert np.abs(inv @ a - np.eye(n)).max() < 1e-8
    sign, mag = np.linalg.slogdet(a)
    got = isle.logdet(a)
    assert abs(got.real - mag) < 1e-10 * max(1.0, abs(mag))
    assert abs(np.exp(1j * got.imag) - sign) < 1e-9
