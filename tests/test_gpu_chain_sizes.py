"""Amplitude and slice chains around the edges of their 64-row, 16-column workgroups, against plain numpy.
An amplitude is a product of n matrices of a state of norm 1: its rounding error is below n chi eps, and the
bar is 1e-12 (complex64 sites are exact in it: the products run on their values in double)."""
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


def build(eng, bonds, precision):
    rng = np.random.default_rng(len(bonds))
    dt = np.complex64 if precision == "mixed" else np.complex128
    s, sites = mps.MpsState(eng, len(bonds) - 1, precision=precision), []
    for k, (cl, cr) in enumerate(zip(bonds[:-1], bonds[1:])):
        a = rng.standard_normal((2 * cl, cr)) + 1j * rng.standard_normal((2 * cl, cr))
        sites.append(np.linalg.qr(a)[0].reshape(cl, 2, cr).astype(dt).astype(np.complex128))
        s.set_site(k, sites[-1])
    return s, sites


@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("count", [1, 15, 63, 64, 65, 130])
@pytest.mark.parametrize("bonds", BONDS)
def test_amplitudes(eng, bonds, count, precision):
    print("amplitudes", bonds, count, precision, flush=True)
    s, sites = build(eng, bonds, precision)
    rng = np.random.default_rng(count)
    p = rng.choice([0.0, 0.05, 0.5, 1.0], size=len(sites))  # sites with one value only, few ones, both
    bits = (rng.random((count, len(sites))) < p).astype(np.int8)
    want = np.empty(count, dtype=np.complex128)
    for i in range(count):
        v = np.ones(1, dtype=np.complex128)
        for k, a in enumerate(sites):
            v = v @ a[:, bits[i, k], :]
        want[i] = v[0]
    got = s.amplitudes(bits)
    assert np.abs(got - want).max() < 1e-12
    assert np.array_equal(s.amplitudes_noalloc(bits), got)
    s.close()


@pytest.mark.parametrize("bonds", BONDS[:4])
def test_slices(eng, bonds):
    print("slices", bonds, flush=True)
    s, sites = build(eng, bonds, "fp64")
    rng = np.random.default_rng(5)
    for _ in range(3):
        spec = rng.choice([-1, -1, 0, 1], size=len(sites))
        v = np.ones((1, 1), dtype=np.complex128)  # open legs: the first site fastest
        for k, a in enumerate(sites):
            v = np.concatenate([v @ a[:, 0, :], v @ a[:, 1, :]]) if spec[k] < 0 else v @ a[:, spec[k], :]
        assert np.abs(s.slice(spec) - v[:, 0]).max() < 1e-12
    s.close()
