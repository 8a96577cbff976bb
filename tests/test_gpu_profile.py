"""Phase times of waves whose gates all run in one workgroup each, which the phases of larger gates do not have."""
import pytest

from tnqvm_amd import circuits as C
from tnqvm_amd import mps

pytestmark = pytest.mark.gpu

PHASES = ("ms_theta", "ms_lq", "ms_jacobi", "ms_split")


@pytest.mark.parametrize("n,chi,small,large", [(10, 16, True, False), (16, 128, True, True)])
def test_every_wave_is_timed(n, chi, small, large):
    print("profile", n, chi, flush=True)
    gates = C.haar_brickwork(n, 10, seed=0x7E5A0C01)
    e = mps.Engine()
    try:
        for timed in (False, True):
            e.set_timing(timed)
            e.profile(reset=True)
            s = mps.MpsState(e, n, cutoff=1e-10, max_bond=chi).run(gates)
            s.flush()
            s.close()
            p = e.profile(reset=True)
            assert (p["ms_other"] > 0.0) == (timed and small)
            assert (sum(p[k] for k in PHASES) > 0.0) == (timed and large)
            assert p["wave_tasks"] == C.count_2q(gates) and p["jacobi_sweeps"] >= p["wave_tasks"]
    finally:
        e.close()
