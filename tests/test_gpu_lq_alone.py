"""A gate's sites are the same to the bit alone and beside wider ones in its wave, at the column counts where the
LQ's panels change from two rows of a lane to one (1024, also reached by the later panels of a wider matrix) and
from one number of columns a lane to the next; and however many lanes the panels are dealt to."""
import numpy as np
import pytest

from tnqvm_amd import mps

pytestmark = pytest.mark.gpu

SIZES = [(66, 130), (100, 300), (130, 130), (70, 1022), (70, 1024), (70, 1026), (1040, 90), (80, 1100), (70, 1536),
         (66, 1538), (66, 2048)]


@pytest.fixture(scope="module")
def eng():
    e = mps.Engine()
    yield e
    e.close()


def planted(eng, m, n):
    rng = np.random.default_rng([m, n])
    a = (rng.standard_normal((m, n)) + 1j * rng.standard_normal((m, n))) / np.sqrt(m * n)
    s = mps.MpsState(eng, 4)
    s.set_site(0, np.ones((1, 2, m // 2)) / m)
    if m <= n:
        s.set_site(1, np.eye(m).reshape(m // 2, 2, m))
        s.set_site(2, a.reshape(m, 2, n // 2))
    else:
        s.set_site(1, a.reshape(m // 2, 2, n))
        s.set_site(2, np.eye(n).reshape(n, 2, n // 2))
    s.set_site(3, np.ones((n // 2, 2, 1)) / n)
    s.apply({"name": "unitary", "qubits": (1, 2), "matrix": np.eye(4)})
    return s


def run(eng, sizes):
    states = [planted(eng, m, n) for m, n in sizes]
    mps.run_waves(states)
    out = [(s.get_site(1), s.get_site(2)) for s in states]
    for s in states:
        s.close()
    return out


def same(a, b):
    return all(np.array_equal(x, y) for x, y in zip(a, b))


def test_same_bits_beside_wider_ones(eng):
    print("lq beside wider ones", flush=True)
    alone = [run(eng, [x])[0] for x in SIZES]
    for beside in (SIZES, SIZES[:5], SIZES[:6] + SIZES[:4], SIZES[2:9]):
        got = run(eng, beside)
        assert [x for x, sites in zip(beside, got) if not same(sites, alone[SIZES.index(x)])] == []


@pytest.mark.parametrize("lanes", [1, 2, 3, 4])
def test_same_bits_on_any_lanes(eng, lanes):
    """64 LQs or more are dealt to lanes."""
    print("lq lanes", lanes, flush=True)
    alone = run(eng, [(66, 130)])[0]
    base = eng.tuning()
    try:
        eng.set_tuning(jacobi_lanes=lanes)
        got = run(eng, [(66, 130)] * 66)
    finally:
        eng.set_tuning(**base)
    assert all([same(sites, alone) for sites in got])
