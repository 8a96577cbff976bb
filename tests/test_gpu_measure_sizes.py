"""Measurements at sizes around the edges of the products' 32 x 16 tiles and 4-wide units, against plain
numpy environments.  A value is a sum over n chained products of bond chi on a state of norm 1, whose
rounding error is below n chi eps times a small factor: the bar is 1e-11."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu

BONDS = [[1, 2, 1], [1, 2, 3, 2, 1], [1, 2, 4, 7, 9, 17, 15, 8, 4, 2, 1], [1, 2, 4, 8, 16, 32, 33, 31, 16, 5, 3, 2, 1],
         [1, 2, 4, 8, 16, 32, 64, 65, 127, 63, 34, 17, 9, 5, 2, 1]]


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def random_sites(bonds, seed, precision):
    rng = np.random.default_rng(seed)
    dt = np.complex64 if precision == "mixed" else np.complex128
    out = []
    for cl, cr in zip(bonds[:-1], bonds[1:]):
        a = rng.standard_normal((2 * cl, cr)) + 1j * rng.standard_normal((2 * cl, cr))
        out.append(np.linalg.qr(a)[0].reshape(cl, 2, cr).astype(dt).astype(np.complex128))
    return out


def state(eng, sites, precision):
    s = mps.MpsState(eng, len(sites), precision=precision)
    for k, a in enumerate(sites):
        s.set_site(k, a)
    return s


def expval(sites, diag):
    e = np.ones((1, 1), dtype=np.complex128)
    for a, d in zip(sites, diag):
        x = np.tensordot(e, a * np.asarray(d).reshape(1, 2, 1), axes=(1, 0))
        e = np.tensordot(a.conj(), x, axes=([0, 1], [0, 1]))
    return e[0, 0].real


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("bonds", BONDS)
def test_observables(eng, bonds, precision):
    print("observables", bonds, precision, flush=True)
    sites = random_sites(bonds, 7 + len(bonds), precision)
    n = len(sites)
    s = state(eng, sites, precision)

    def diag(qs):
        return [(1.0, -1.0) if qs.count(k) % 2 else (1.0, 1.0) for k in range(n)]

    z = np.array([expval(sites, diag([k])) for k in range(n)])
    pairs = [(a, b) for a in range(n) for b in range(n) if (a * 5 + b * 3) % 4 == 0]  # both orders, repeats, i == i
    zz = np.array([expval(sites, diag([a, b])) for a, b in pairs])
    d = np.random.default_rng(3).standard_normal((n, 2))
    assert np.abs(s.expval_z_all() - z).max() < 1e-11
    assert np.abs(s.expval_zz(pairs) - zz).max() < 1e-11
    assert abs(s.norm() - expval(sites, diag([]))) < 1e-11
    assert abs(s.expval_z_parity(range(0, n, 2)) - expval(sites, diag(list(range(0, n, 2))))) < 1e-11
    assert abs(s.expval_diag(d) / np.abs(d).max(1).prod() - expval(sites, d) / np.abs(d).max(1).prod()) < 1e-11
    qs = [n - 1, 0]
    want = np.zeros(4)
    for x in range(4):
        pr = {qs[0]: x & 1, qs[1]: x >> 1}
        want[x] = expval(sites, [(1.0, 1.0) if k not in pr else (float(pr[k] == 0), float(pr[k] == 1)) for k in range(n)])
    assert np.abs(s.outcome_probabilities(qs) - want).max() < 1e-11
    s.close()


@pytest.mark.parametrize("measured", [[0], [9], [0, 1, 2, 3, 4, 5, 6, 7, 8, 9], [1, 3, 4, 8], [7, 8], [2, 9]])
def test_sampling_marginals(eng, measured):
    """Every site measured, some traced before and between (environments held as factors or densely):
    the strings of sequential marginals of the dense state under the same draws."""
    print("sampling", measured, flush=True)
    bonds = [1, 2, 4, 8, 15, 17, 9, 8, 4, 2, 1]
    sites = random_sites(bonds, 11, "fp64")
    v = sites[0].reshape(2, -1)
    for a in sites[1:]:
        v = np.tensordot(v, a, axes=(v.ndim - 1, 0))
    p = np.abs(v.reshape((2,) * 10)) ** 2
    marg = p.sum(axis=tuple(q for q in range(10) if q not in measured))
    shots, k = 37, len(measured)
    draws = np.random.default_rng(5).random((shots, k))
    want = []
    for t in range(shots):
        bits, given = "", 1.0
        for i in range(k):
            m = marg[tuple(int(b) for b in bits)]
            m = m.reshape(2, -1).sum(1) / given
            b = 0 if draws[t, i] <= m[0] else 1
            given *= m[b]
            bits += str(b)
        want.append(bits)
    s = state(eng, sites, "fp64")
    assert s.sample_sequential(measured, draws) == want
    s.close()
