"""Qubits that MpsState.outcome_probabilities takes and refuses, without a device: the call into the library is
replaced by one that records them."""
import numpy as np
import pytest

from tnqvm_amd import mps


class State(mps.MpsState):
    def __init__(self, n):
        self.n, self.h, self.e = n, None, None


class Lib:
    def hipmps_outcome_probabilities(self, h, q, k, out):
        self.q = [q[i] for i in range(k)]
        return 0


@pytest.fixture
def taken(monkeypatch):
    lib = Lib()
    monkeypatch.setattr(mps, "lib", lambda: lib)

    def call(qubits):
        lib.q = None
        return State(5).outcome_probabilities(qubits), lib.q

    return call


@pytest.mark.parametrize("qubits,want", [([], []), ([3], [3]), ((0, 4), [0, 4]), ([-1, -5], [4, 0]), ([2, 2], [2, 2]),
                                         (np.array([1, 3]), [1, 3]), ([np.int64(2), True], [2, 1]), (range(5), [0, 1, 2, 3, 4])])
def test_taken(taken, qubits, want):
    out, got = taken(qubits)
    assert got == want and out.shape == (1 << len(want),)


@pytest.mark.parametrize("qubits,error", [([5], IndexError), ([-6], IndexError), ([1 << 40], IndexError), ([-1 << 40], IndexError),
                                          ([1.0], (IndexError, TypeError)), (np.array([1.0, 2.0]), (IndexError, TypeError)),
                                          ([0.5], (IndexError, TypeError)), (["1"], (IndexError, TypeError)),
                                          ([[0], [1]], (IndexError, TypeError)), ([None], (IndexError, TypeError)),
                                          (list(range(17)), ValueError)])
def test_refused(taken, qubits, error):
    with pytest.raises(error):
        taken(qubits)


def test_arrays_as_elements(taken, monkeypatch):
    """An integer array as an element stands for its qubits together, as it indexes a diagonal."""
    seen = []
    monkeypatch.setattr(State, "expval_diag", lambda self, d: seen.append(list(d)) or 0.0)
    taken([np.array([0, 2])])
    assert seen == [[1, 0, 1, 1, 1, 0, 1, 1, 1, 1], [0, 1, 1, 1, 0, 1, 1, 1, 1, 1]]
