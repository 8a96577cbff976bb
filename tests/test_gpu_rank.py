"""Bonds of a state whose Schmidt ranks stay low for a while, against the FP64 oracle MPS under the same
truncation.  Rounding residue of a numerically zero singular value that a split keeps (the index below the
cutoff) and that comes back in the next theta' above the cutoff would make them grow."""
import pytest

from oracle import oracle as O
from tnqvm_amd import circuits as C
from tnqvm_amd import mps

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


@pytest.mark.parametrize("n,count", [(14, 40), (14, 60), (14, 80), (14, 100), (20, 60), (20, 90)])
def test_bonds_follow_the_ranks(eng, n, count):
    print("ranks", n, count, flush=True)
    gates = C.qaoa_maxcut(n, 4, seed=0x7E5A0301)[0][:count]
    ref = O.Mps(n, cutoff=1e-12, max_bond=0)
    for g in gates:
        ref.apply(g)
    s = mps.MpsState(eng, n, cutoff=1e-12).run(gates)
    s.flush()
    assert list(s.bonds()) == list(ref.bonds())
    s.close()
