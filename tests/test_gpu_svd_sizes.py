"""The SVD at the edges of its kernels' ranges: sizes around a multiple of the 16-row blocks, of the
32-row pairs and of the block counts at which the sweeps' orderings change, against a spectrum known
by construction (12 decades) at the suite's bar for known spectra, 1e-12."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def graded(m, n, seed, decades=12.0):
    rng = np.random.default_rng(seed)
    k = min(m, n)
    u = np.linalg.qr(rng.standard_normal((m, k)) + 1j * rng.standard_normal((m, k)))[0]
    v = np.linalg.qr(rng.standard_normal((n, k)) + 1j * rng.standard_normal((n, k)))[0]
    s = np.logspace(0.0, -decades, k)
    return (u * s) @ v.conj().T, s


@pytest.mark.parametrize("m,n", [(2, 2), (4, 2), (2, 34), (16, 16), (18, 14), (32, 32), (30, 66), (34, 34), (64, 62),
                                 (66, 64), (66, 130), (96, 96), (98, 100), (130, 128), (160, 96), (224, 226), (226, 240),
                                 (256, 258), (514, 130), (516, 514)])
def test_svd_sizes(eng, m, n):
    print("svd", m, n, flush=True)
    a, sref = graded(m, n, seed=m + 3 * n)
    cl, cr = m // 2, n // 2
    s = mps.MpsState(eng, 4)
    s.set_site(0, np.ones((1, 2, cl)) / np.sqrt(2 * cl))
    s.set_site(1, a.reshape(cl, 2, n))
    s.set_site(2, np.eye(n).reshape(n, 2, cr))
    s.set_site(3, np.ones((cr, 2, 1)) / np.sqrt(2 * cr))
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    s.flush()
    left, right = s.get_site(1).reshape(m, -1), s.get_site(2).reshape(-1, n)
    sig = (np.abs(left) ** 2).sum(0)
    s.close()
    assert len(sig) == min(m, n)
    assert np.abs(sig - sref).max() < 1e-12
    assert np.abs(left @ right - a).max() < 1e-12
