"""Finite sites whose theta' overflows in one column or row only: HIPMPS_E_NUMERIC, whichever side of the LQ's
diagonal the NaN lies on, for gates of one workgroup (small) and for larger ones."""
import numpy as np
import pytest

from tnqvm_amd import _capi as capi
from tnqvm_amd import circuits as C
from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def planted(eng, left, right):
    """Sites 1 and 2 of 4 with the bonds they need on either side; a 2-qubit gate between them is queued."""
    s = mps.MpsState(eng, 4, precision="fp64")
    cl, cr = left.shape[0], right.shape[2]
    s.set_site(0, np.ones((1, 2, cl)) / np.sqrt(2 * cl))
    s.set_site(1, left)
    s.set_site(2, right)
    s.set_site(3, np.ones((cr, 2, 1)) / np.sqrt(2 * cr))
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": C.haar_unitary(np.random.default_rng(5), 4)})
    return s


# theta' of 2 rows and 2 width columns, or the other way round (50: also with the larger LDS)
@pytest.mark.parametrize("side", ["right", "left"])
@pytest.mark.parametrize("place", [0, 1, -1])
@pytest.mark.parametrize("width", [4, 8, 32, 50])
def test_overflow_in_one_place(eng, width, place, side):
    print("overflow in one place", width, place, side, flush=True)
    one = np.full((1, 2, 1), 1e10, dtype=np.complex128)
    wide = np.ones((1, 2, width), dtype=np.complex128)
    wide[0, :, place] = 1e300
    s = planted(eng, one, wide) if side == "right" else planted(eng, wide.transpose(2, 1, 0), one)
    with pytest.raises(capi.HipMpsError) as ei:
        s.flush()
    assert ei.value.code == capi.HIPMPS_E_NUMERIC
    s.close()


@pytest.mark.parametrize("bond,width", [(2, 8), (8, 8), (16, 60), (40, 60)])
def test_overflow_in_the_last_row(eng, bond, width):
    """The last row of theta', where an LQ has no row below to carry the NaN on to."""
    print("overflow in the last row", bond, width, flush=True)
    rng = np.random.default_rng(bond)
    left = rng.standard_normal((bond, 2, bond)) + 0j
    right = rng.standard_normal((bond, 2, width)) + 0j
    left[:, :, -1] = 0.0
    left[-1, 1, -1] = 1e200  # meets the last row of the right site alone
    right[-1, 1, -1] = 1e200
    s = mps.MpsState(eng, 4, precision="fp64")
    s.set_site(0, np.ones((1, 2, bond)))
    s.set_site(1, left)
    s.set_site(2, right)
    s.set_site(3, np.ones((width, 2, 1)))
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    with pytest.raises(capi.HipMpsError) as ei:
        s.flush()
    assert ei.value.code == capi.HIPMPS_E_NUMERIC
    s.close()
