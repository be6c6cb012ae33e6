"""GPU: the volume average at the edges of its blocks (64 elements a partial, 256 a row of four), against the oracle.

Both add the 8 nelem Gauss-point stresses in some order: each is within 8 nelem rounding errors of the mean magnitude,
for which the mean of the elements' averages stands (no larger)."""
import numpy as np
import pytest

from oracle import bindings as ob

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mp():
    import micropp_amd

    micropp_amd.load()
    if not micropp_amd.gpu_available():
        pytest.skip("no HIP device")
    return micropp_amd


@pytest.mark.parametrize("law", [((0, 1e6, 0.3), (0, 1e7, 0.25)), ((1, 1e6, 0.3, 1e5, 1e4), (0, 1e7, 0.25))],
                         ids=["elastic", "j2"])
@pytest.mark.parametrize("elems", [(1, 1, 1), (7, 3, 3), (8, 8, 1), (13, 5, 1), (17, 15, 1), (16, 16, 1), (257, 1, 1),
                                   (11, 10, 12), (33, 32, 31)], ids=lambda s: "x".join(map(str, s)))
def test_average_stress(mp, oracle, elems, law):
    size = tuple(n + 1 for n in elems)
    laws = law + law[1:]
    r = mp.Rve(size, 1, (0.3,) * 4, [mp.material(*m) for m in laws])
    o = oracle.rve(size, 1, (0.3,) * 4, [ob.material(*m) for m in laws])
    u = np.random.default_rng(sum(elems)).normal(0, 4e-3, r.nrow)
    s, du = mp.Solver(r), mp.DeviceArray.from_numpy(u)
    sig, ref = s.ave_stress(du), o.ave_stress(u)
    mean = np.abs(s.elem_fields(du)[1]).reshape(-1, 6).mean(axis=0)
    assert (np.abs(sig - ref) <= 2 * 8 * r.nelem * 2.3e-16 * np.maximum(mean, np.abs(ref))).all()
