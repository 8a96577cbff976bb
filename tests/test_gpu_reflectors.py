"""The lengths that the LQ's reflectors give, to working precision.

theta' has orthogonal rows of disjoint supports and equal length, so that every reflector acts on one row, no row
rotates, and every singular value is that length.  Its square, 3.6872878, is an argument at which the hardware's
reciprocal root refined by one Newton step is 19 eps off.  A value passes through a sum of squares, one reflector
(two in gates of 64 rows and more, whose LQ is a double one, and the application of both), a norm and its root: fewer
than 20 and 40 roundings of eps / 2, hence the bars of 10 and 20 eps."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


@pytest.mark.parametrize("transposed", [False, True])
@pytest.mark.parametrize("scale", [1, 2])
@pytest.mark.parametrize("r,c", [(2, 16), (8, 16), (16, 32), (32, 64), (64, 128), (66, 132), (100, 200), (66, 2046),
                                 (66, 2200)])
def test_length_of_rows(eng, r, c, scale, transposed):
    print("length of rows", r, c, scale, transposed, flush=True)
    x = 3.6872878328006582 * 4.0 ** scale
    w = c // r
    t = np.zeros((r, c), dtype=np.complex128)
    for i in range(r):
        t[i, w * i:w * i + w] = np.sqrt(x / w) * 1j ** (np.arange(w) + i)
    sigma = np.sqrt((np.abs(t) ** 2).sum(1))
    if transposed:
        t = t.T
    m, n = t.shape
    s = mps.MpsState(eng, 4, cutoff=1e-10)
    s.set_site(0, np.ones((1, 2, m // 2)) / m)
    if transposed:
        s.set_site(1, t.reshape(m // 2, 2, n))
        s.set_site(2, np.eye(n).reshape(n, 2, n // 2))
    else:
        s.set_site(1, np.eye(m).reshape(m // 2, 2, m))
        s.set_site(2, t.reshape(m, 2, n // 2))
    s.set_site(3, np.ones((n // 2, 2, 1)) / n)
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    s.flush()
    left, right = s.get_site(1).reshape(m, -1), s.get_site(2).reshape(-1, n)
    s.close()
    assert left.shape[1] == r
    bar = (20 if r >= 64 else 10) * np.finfo(np.float64).eps
    assert np.abs((np.abs(left) ** 2).sum(0) / sigma - 1.0).max() < bar
    assert np.abs((np.abs(right) ** 2).sum(1) / sigma - 1.0).max() < bar
    assert np.abs(left @ right - t).max() < bar * sigma[0]
