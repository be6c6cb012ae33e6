"""GPU: the element kernels at the edges of their blocks, bit for bit against the oracle.

Grids without an interior node, of one element, of fewer elements than a block and with a remainder of elements,
rows and Gauss points, with a yielded history and without; all three phases, one of them elastic beside a
nonlinear matrix (both branches of the tangent in one block)."""
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


LAWS = {"elastic": ((0, 1e6, 0.3), (0, 1e7, 0.25), (0, 3e6, 0.2)),
        "j2": ((1, 1e6, 0.3, 1e5, 1e4), (0, 1e7, 0.25), (1, 3e6, 0.2, 1e4, 3e3)),
        "damage": ((2, 1e6, 0.3, 0.0, 0.0, 1e5), (0, 1e7, 0.25), (2, 3e6, 0.2, 0.0, 0.0, 1e5))}


@pytest.mark.parametrize("law", list(LAWS))
@pytest.mark.parametrize("size", [(2, 2, 2), (3, 3, 3), (2, 9, 4), (23, 3, 5), (12, 11, 13)],
                         ids=lambda s: "x".join(map(str, s)))
def test_element_kernels_bitwise(mp, oracle, size, law):
    gm = [mp.material(*m) for m in LAWS[law]]
    om = [ob.material(*m) for m in LAWS[law]]
    geo = (0.3,) * 4
    r = mp.Rve(size, 1, geo, gm)
    s = mp.Solver(r)
    o = oracle.rve(size, 1, geo, om)
    rng = np.random.default_rng(sum(size))
    u = rng.normal(0, 4e-3, r.nrow)
    du, db, dv = mp.DeviceArray.from_numpy(u), mp.DeviceArray(r.nrow), mp.DeviceArray(r.nvars)
    history = None
    for _ in range(2):  # from no history, then from the history that leaves
        old = None if history is None else mp.DeviceArray.from_numpy(history)
        s.assembly_mat(du, old)
        assert np.array_equal(s.ell()[1], o.assembly_mat(u, history))
        norm = s.assembly_rhs(du, old, db)
        b, n = o.assembly_rhs(u, history)
        assert np.array_equal(db.numpy(), b) and abs(norm - n) <= 1e-13 * n
        # the volume average sums 8 nelem terms of one sign and scale at most: n rounding errors of the largest
        sig, ref = s.ave_stress(du, old), o.ave_stress(u, history)
        assert np.abs(sig - ref).max() <= 8 * r.nelem * 2.3e-16 * max(1.0, np.abs(ref).max()) * 1e3
        nl = s.vars_new(du, old, dv)
        new, nlo = o.vars_new(u, history)
        assert nl == nlo and np.array_equal(dv.numpy(), new)
        history = new
