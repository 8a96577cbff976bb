"""Sampling with many traced qubits ahead of the last measured one: a factored left environment would have a row per
configuration of theirs, so the shots take dense ones, which stay small."""
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


def test_long_traced_tail():
    print("long traced tail", flush=True)
    rng = np.random.default_rng(8)
    n, tail, shots = 14, 17, 100
    bonds = [min(1 << min(k, n - k), 64) for k in range(n + 1)]
    block = []
    for cl, cr in zip(bonds[:-1], bonds[1:]):
        a = rng.standard_normal((2 * cl, cr)) + 1j * rng.standard_normal((2 * cl, cr))
        block.append(np.linalg.qr(a)[0].reshape(cl, 2, cr))
    one = np.array([0.6, 0.8j]).reshape(1, 2, 1)
    draws = rng.random(shots * (n + 1))
    e = mps.Engine()
    try:
        out = []
        for traced in (0, tail):  # the traced qubits are in a product with the others: the strings are the same
            sites = block + [one] * (traced + 1)
            s = mps.MpsState(e, len(sites))
            for k, a in enumerate(sites):
                s.set_site(k, a)
            s.flush()
            before = free_bytes()
            out.append(s.sample_sequential(list(range(n)) + [len(sites) - 1], draws))
            held = before - free_bytes()
            s.close()
        assert out[0] == out[1]
        assert held < 128 << 20
    finally:
        e.close()
