"""GPU: the multi-RHS solver's FP32 operator as a stencil dictionary.

Runs of 62 nodes, four per block: sizes whose node counts lie just below, at and just above whole runs
and blocks, x-lines shorter and longer than a run, and three phases (every digit of a stencil's code).
Bar: sigma and ctan within 1e-6 of the FP64 path, both solved to 1e-8 of the start residual.
"""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu


@pytest.fixture(scope="module")
def mp():
    import micropp_amd

    micropp_amd.load()
    if not micropp_amd.gpu_available():
        pytest.skip("no HIP device")
    return micropp_amd


def rel(a, b):
    return np.abs(np.asarray(a) - np.asarray(b)).max() / np.abs(np.asarray(b)).max()


@pytest.mark.parametrize("size, K", [((5, 5, 10), 8), ((4, 4, 31), 12), ((31, 4, 4), 12), ((3, 31, 8), 8),
                                     ((62, 4, 5), 8), ((64, 5, 4), 16), ((7, 9, 63), 8), ((70, 3, 3), 8)])
def test_stencil_operator_three_phases(mp, size, K):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 3e6, 0.2)]
    strains = np.random.default_rng(sum(size)).uniform(-5e-3, 5e-3, (2, 6))
    r = mp.Rve(size, mp.MIC3D_8, (0.1, 0.0, 0.0, 0.0), mats)
    sig, ctan, _, resid, ok = mp.homogenize_mixed(mp.MSolver(r, K), strains)
    assert ok and resid.max() < 1e-8
    m = mp.Micropp3(size, mp.MIC3D_8, (0.1, 0.0, 0.0, 0.0), mats, ngp=2, coupling=[mp.FE_ONE_WAY] * 2, lin_stress=0,
                    cg_rel_tol=1e-8, cg_max_its=4000)
    for g in range(2):
        m.set_strain(g, strains[g])
    m.homogenize()
    assert rel(sig, np.array([m.get_stress(g) for g in range(2)])) < 1e-6
    assert rel(ctan, m.ctan_lin()) < 1e-6
