"""Noise channels at sizes around the edges of the one-workgroup kernel (64 rows, its two LDS variants, both
orientations of the rows), against numpy.  The site before a channel is read back, so one channel's error is
measured: rho = sum_k A_k A_k^H of the new site differs from numpy's (kept rows of an SVD) by the rounding
of about 10 sweeps of 64 rotations on entries of a site of norm 1, below 1e-12 in double; in float the site
is rounded to 2^-24 and the sweeps stop at a relative inner product of 1e-7 or so, below 1e-5."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def channel(rng, n_ops):
    q = np.linalg.qr(rng.standard_normal((2 * n_ops, 2)) + 1j * rng.standard_normal((2 * n_ops, 2)))[0]
    return q.reshape(n_ops, 2, 2)


def expected(a, ops, kap):
    cl, _, _, cr = a.shape
    x = np.einsum("opq,lqkr->kolpr", ops, a).reshape(kap * len(ops), 2 * cl * cr)
    _, sv, vh = np.linalg.svd(x, full_matrices=False)
    below = np.nonzero(sv * sv < 1e-9)[0]
    keep = max(1, min(int(below[0]) if len(below) else len(sv), 2 * cl * cr, 2 * kap))
    y = sv[:keep, None] * vh[:keep]
    return keep, y.T @ y.conj()  # over (l, p, r)


# (left bond, right bond, operators of each channel in turn)
CASES = [(1, 1, [1, 2, 2]), (1, 2, [2, 3, 16]), (2, 2, [4, 4, 4]), (2, 3, [2, 2, 3, 5]), (1, 5, [3, 3, 3, 5, 2]),
         (4, 4, [2, 4, 4, 4, 16]), (3, 5, [4, 4, 4, 2]), (4, 8, [4, 4, 4]), (5, 7, [4, 4, 4]), (3, 11, [16, 2, 4])]


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("cl,cr,ops", CASES)
def test_channels(eng, cl, cr, ops, precision):
    print("channels", cl, cr, ops, precision, flush=True)
    rng = np.random.default_rng(100 * cl + cr)
    s = mps.MpsState(eng, 3, precision=precision)
    for k, (p, q) in enumerate([(1, cl), (cl, cr), (cr, 1)]):
        a = rng.standard_normal((p, 2, q)) + 1j * rng.standard_normal((p, 2, q))
        s.set_site(k, a / np.linalg.norm(a))
    for n_ops in ops:
        a = s.get_site(1)
        a = a.reshape(cl, 2, -1, cr)
        kap = a.shape[2]
        k = channel(rng, n_ops)
        s.apply_kraus(1, k)
        s.flush()
        b = s.get_site(1).reshape(cl, 2, -1, cr)
        keep, rho = expected(a, k, kap)
        assert b.shape[2] == keep
        y = b.transpose(2, 0, 1, 3).reshape(keep, -1)
        assert np.abs(y.T @ y.conj() - rho).max() < (1e-12 if precision == "fp64" else 1e-5)
    s.close()
