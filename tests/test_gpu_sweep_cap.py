"""Sweep caps far above what an SVD takes: nothing is held or cleared for sweeps that do not run, results are those
of the default cap, and a gate that never converges ends at the cap."""
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


def planted(eng, m):
    rng = np.random.default_rng(m)
    a = (rng.standard_normal((m, m)) + 1j * rng.standard_normal((m, m))) / m
    s = mps.MpsState(eng, 4)
    s.set_site(0, np.ones((1, 2, m // 2)) / m)
    s.set_site(1, np.eye(m).reshape(m // 2, 2, m))
    s.set_site(2, a.reshape(m, 2, m // 2))
    s.set_site(3, np.ones((m // 2, 2, 1)) / m)
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    return s, a


def test_large_cap_costs_nothing():
    print("large sweep cap", flush=True)
    out, held = [], []
    for cap in (0, 100_000_000):
        e = mps.Engine(jacobi_max_sweeps=cap)
        try:
            states = [planted(e, 70)[0] for _ in range(4)]
            before = free_bytes()
            mps.run_waves(states)
            held.append(before - free_bytes())
            out.append([s.get_site(1) for s in states])
        finally:
            e.close()
    assert held[1] < held[0] + (64 << 20)
    assert all(np.array_equal(a, b) for a, b in zip(*out))


@pytest.mark.parametrize("cap", [1, 2, 63, 64, 65, 66, 130])
def test_ends_at_the_cap(cap):
    """A tolerance that no SVD reaches: as many sweeps as the cap says."""
    print("ends at the cap", cap, flush=True)
    e = mps.Engine(jacobi_max_sweeps=cap, jacobi_tol=1e-30)
    try:
        s, a = planted(e, 70)
        with pytest.raises(capi.HipMpsError) as ei:
            s.flush()
        assert ei.value.code == capi.HIPMPS_E_CONVERGENCE
        st = s.stats()
        assert st["jacobi_sweeps_max"] == cap and st["svds_nonconverged"] == 1
        s.close()
    finally:
        e.close()


@pytest.mark.parametrize("m,cap,ends", [(4, 40, 40), (4, 1000, 1000), (4, 20000, 1000)])
def test_one_launch_is_bounded(m, cap, ends):
    """A gate in one workgroup sweeps within one launch, which has to end soon whatever the cap."""
    print("one launch is bounded", m, cap, flush=True)
    e = mps.Engine(jacobi_max_sweeps=cap, jacobi_tol=1e-30)
    try:
        s, a = planted(e, m)
        with pytest.raises(capi.HipMpsError) as ei:
            s.flush()
        assert ei.value.code == capi.HIPMPS_E_CONVERGENCE
        assert s.stats()["jacobi_sweeps_max"] == ends
        s.close()
    finally:
        e.close()
