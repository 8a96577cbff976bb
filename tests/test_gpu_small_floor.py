"""Singular values below 1e-15 of the largest in a gate of one workgroup: the truncation rule counts them as it does
in larger gates (the index that falls below the cutoff is kept, those at or above it too), and they are in the sites
when the cutoff leaves them."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def split(eng, sigma, rows, cols, cutoff):
    """theta' (rows x cols) with the given values on its diagonal, through the identity gate; its new bond and sites."""
    t = np.zeros((rows, cols), dtype=np.complex128)
    np.fill_diagonal(t, sigma)
    s = mps.MpsState(eng, 4, cutoff=cutoff)
    s.set_site(0, np.ones((1, 2, rows // 2)) / rows)
    s.set_site(1, t.reshape(rows // 2, 2, cols))
    s.set_site(2, np.eye(cols).reshape(cols, 2, cols // 2))
    s.set_site(3, np.ones((cols // 2, 2, 1)) / cols)
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    s.flush()
    out = int(s.bonds()[2]), s.get_site(1).reshape(rows, -1), s.get_site(2).reshape(-1, cols)
    s.close()
    return out


# 80 x 80 and 80 x 90 take the path of larger gates
@pytest.mark.parametrize("rows,cols", [(4, 4), (8, 6), (10, 64), (64, 64), (80, 80), (80, 90)])
@pytest.mark.parametrize("cutoff", [0.0, 2.2250738585072014e-308, 3e-22, 3e-18])
def test_values_below_the_floor(eng, rows, cols, cutoff):
    print("below the floor", rows, cols, cutoff, flush=True)
    k = min(rows, cols)
    # 1, then 1e-16 10^-j
    sigma = np.array([1.0] + [10.0 ** -min(16 + j, 30) for j in range(k - 1)])
    above = int((sigma >= cutoff).sum())
    want = min(k, above + 1) if above < k else k
    bond, left, right = split(eng, sigma, rows, cols, cutoff)
    assert bond == want
    got = np.diag(left @ right)[:above]
    assert np.abs(got / sigma[:above] - 1.0).max() < 1e-12
