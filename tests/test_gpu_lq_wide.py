"""A theta' of more than 2^28 elements through the LQ, whose rows lie more than 4 GiB apart: 80 x 2^22, so that the
last panel's 16 rows start at element 2^28."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


def test_rows_past_4_gib():
    print("rows past 4 GiB", flush=True)
    cl, cm, cr = 40, 2, 1 << 21
    rng = np.random.default_rng(17)
    left = rng.standard_normal((cl, 2, cm)) + 1j * rng.standard_normal((cl, 2, cm))
    right = np.empty((cm, 2, cr), dtype=np.complex128)
    right.real = rng.standard_normal(right.shape)
    right.imag = rng.standard_normal(right.shape)
    left /= np.linalg.norm(left)
    right /= np.linalg.norm(right)
    e = mps.Engine()
    try:
        s = mps.MpsState(e, 4, cutoff=1e-10, max_bond=cm)
        s.set_site(0, np.full((1, 2, cl), 1.0))
        s.set_site(1, left)
        s.set_site(2, right)
        s.set_site(3, np.full((cr, 2, 1), 1.0))
        s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
        s.flush()  # raises when the SVD has not converged
        a, b = s.get_site(1).reshape(2 * cl, cm), s.get_site(2).reshape(cm, 2 * cr)
        s.close()
    finally:
        e.close()
    # rank cm: nothing is truncated.  Rows and columns of theta' across the whole range, at the suite's 1e-12 of
    # its norm (which is below 1)
    cols = np.unique(np.concatenate([np.arange(64), rng.integers(0, 2 * cr, 4096), 2 * cr - 1 - np.arange(64)]))
    want = left.reshape(2 * cl, cm) @ right.reshape(cm, 2 * cr)[:, cols]
    assert np.abs(a @ b[:, cols] - want).max() < 1e-12
    # isometries times sqrt(sigma) on both sides: the sites' Gram matrices are diag(sigma)
    ga, gb = a.conj().T @ a, b @ b.conj().T
    assert np.abs(ga - np.diag(np.diag(ga))).max() < 1e-12 and np.abs(np.diag(ga) - np.diag(gb)).max() < 1e-12
