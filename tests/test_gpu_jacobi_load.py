"""Many SVDs in one wave, so that a Jacobi round has more than one workgroup per CU (four waves each), and
few (eight waves each), against a spectrum known by construction at the suite's bar for it, 1e-12."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


@pytest.mark.parametrize("count,m,n", [(2, 130, 128), (51, 130, 162), (52, 162, 130), (72, 128, 128)])
def test_many_svds(eng, count, m, n):
    print("svds", count, m, n, flush=True)
    rng = np.random.default_rng(count + m)
    k = min(m, n)
    u = np.linalg.qr(rng.standard_normal((m, k)) + 1j * rng.standard_normal((m, k)))[0]
    v = np.linalg.qr(rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k)))[0]
    sref = np.logspace(0.0, -12.0, k)
    cl, cr = m // 2, n // 2
    states, mats = [], []
    for i in range(count):  # the same spectrum, rows and columns turned
        a = (np.roll(u, i, axis=0) * sref) @ np.roll(v, 3 * i, axis=0).conj().T
        s = mps.MpsState(eng, 4)
        s.set_site(0, np.ones((1, 2, cl)) / np.sqrt(2 * cl))
        s.set_site(1, a.reshape(cl, 2, n))
        s.set_site(2, np.eye(n).reshape(n, 2, cr))
        s.set_site(3, np.ones((cr, 2, 1)) / np.sqrt(2 * cr))
        s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
        states.append(s)
        mats.append(a)
    mps.run_waves(states)
    for s, a in zip(states, mats):
        left, right = s.get_site(1).reshape(m, -1), s.get_site(2).reshape(-1, n)
        assert left.shape[1] == k
        assert np.abs((np.abs(left) ** 2).sum(0) - sref).max() < 1e-12
        assert np.abs(left @ right - a).max() < 1e-12
        s.close()


def test_result_independent_of_load(eng):
    """A gate's sites are the same to the bit alone and in a wave that fills the chip."""
    print("load", flush=True)
    rng = np.random.default_rng(9)
    m, n = 130, 200
    a = rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))
    out = []
    for count in (1, 60):
        states = []
        for i in range(count):
            s = mps.MpsState(eng, 4)
            s.set_site(0, np.ones((1, 2, m // 2)) / m)
            s.set_site(1, np.roll(a, i, axis=1).reshape(m // 2, 2, n))
            s.set_site(2, np.eye(n).reshape(n, 2, n // 2))
            s.set_site(3, np.ones((n // 2, 2, 1)) / n)
            s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
            states.append(s)
        mps.run_waves(states)
        out.append((states[0].get_site(1), states[0].get_site(2)))
        for s in states:
            s.close()
    assert np.array_equal(out[0][0], out[1][0]) and np.array_equal(out[0][1], out[1][1])
