"""<Z> and <ZZ> of states too large to keep every site's intermediate: the environments of one side are kept
instead, and the results are those of the other form."""
import ctypes

import numpy as np
import pytest

from tnqvm_amd import _capi as capi
from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


def free_bytes():
    free, total = ctypes.c_size_t(), ctypes.c_size_t()
    assert capi.lib().hipMemGetInfo(ctypes.byref(free), ctypes.byref(total)) == 0
    return free.value


def sites(bonds, seed):
    rng = np.random.default_rng(seed)
    made = {}
    for cl, cr in zip(bonds[:-1], bonds[1:]):
        if (cl, cr) not in made:
            made[cl, cr] = (rng.standard_normal((cl, 2, cr)) + 1j * rng.standard_normal((cl, 2, cr))) / np.sqrt(4 * cl)
        yield made[cl, cr]


def state(eng, bonds, seed, precision="fp64"):
    s = mps.MpsState(eng, len(bonds) - 1, precision=precision)
    for k, a in enumerate(sites(bonds, seed)):
        s.set_site(k, a)
    return s


def test_workspace_of_a_large_state():
    """100 qubits at bond 1024: 2.8 GB of sites; all right environments are 1.4 GB.  Kept intermediates of both sides
    were 5.5 GB and a quarter more."""
    print("workspace of a large state", flush=True)
    n = 100
    bonds = [min(1 << min(k, n - k, 20), 1024) for k in range(n + 1)]
    e = mps.Engine()
    try:
        s = state(e, bonds, 3)
        norm = s.norm()
        before = free_bytes()
        z = s.expval_z_all()
        zz = s.expval_zz([(20, 60), (33, 34), (5, 5)])
        held = before - free_bytes()
        assert held < 3 << 30
        # a diagonal's own sweep keeps nothing; 100 products of bond 1024: below 1e-10 of the norm
        for q in (0, 1, 20, 51, 99):
            assert abs(z[q] - s.expval_z_parity([q])) < 1e-10 * norm
        assert abs(zz[0] - s.expval_z_parity([20, 60])) < 1e-10 * norm
        assert abs(zz[1] - s.expval_z_parity([33, 34])) < 1e-10 * norm
        assert abs(zz[2] - norm) < 1e-10 * norm
    finally:
        e.close()


# as test_gpu_measure_sizes: the bar for sums of n chained products of bond chi on a state of norm 1 is 1e-11
BONDS = [[1, 1], [1, 2, 1], [1, 2, 4, 3, 2, 1], [1, 2, 4, 8, 16, 33, 40, 35, 16, 8, 4, 2, 1], [1, 64, 65, 34, 100, 1]]


@pytest.mark.parametrize("kraus", [False, True])
@pytest.mark.parametrize("precision", ["fp64", "mixed"])
@pytest.mark.parametrize("bonds", BONDS)
def test_both_forms_agree(monkeypatch, bonds, precision, kraus):
    print("both forms", bonds, precision, kraus, flush=True)
    n = len(bonds) - 1
    rng = np.random.default_rng(4)
    ops = [np.linalg.qr(rng.standard_normal((6, 2)) + 1j * rng.standard_normal((6, 2)))[0][2 * k:2 * k + 2] for k in range(3)]
    pairs = [(a, b) for a in range(n) for b in range(n) if (a * 5 + b * 3) % 4 != 1]
    out = []
    for keep in (None, "0"):
        if keep is not None:
            monkeypatch.setenv("HIPMPS_TEST_ENV_KEEP_BYTES", keep)
        e = mps.Engine()
        try:
            s = state(e, bonds, 11, precision)
            if kraus:
                for q in range(n):
                    s.apply_kraus(q, ops)
            norm = s.norm()
            out.append((norm, s.expval_z_all(), s.expval_zz(pairs), s.expval_zz(pairs[-1:]), s.expval_zz([(0, 0)])))
            s.close()
        finally:
            e.close()
    for a, b in zip(*out):
        assert np.abs(np.asarray(a) - np.asarray(b)).max() < 1e-11 * out[0][0]
