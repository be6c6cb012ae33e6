"""GPU: the multi-RHS preconditioner at the edge between two levels and three.

Coarse elements 1 to 3 wide right above the fine grid (sides of 4 to 26 elements), the largest and smallest coarse
solves of its three load depths (3 to 2187 DOFs: at most 256, 512 and more columns), a remainder of
rows and columns in its 16-wide tiles, and 4 to 16 fields.
Bar, as for the other preconditioners: sigma and ctan within 1e-6 of the Jacobi-preconditioned solve (both to 1e-8 of
the start residual), with fewer inner iterations."""
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


@pytest.mark.parametrize("size, K", [((5, 5, 5), 8), ((7, 10, 8), 12), ((9, 9, 9), 16), ((13, 13, 13), 12),
                                     ((19, 17, 18), 8), ((19, 19, 19), 16), ((21, 20, 21), 12), ((23, 23, 23), 12), ((27, 27, 27), 8),
                                     ((28, 27, 26), 8)])
def test_two_levels_against_jacobi(mp, monkeypatch, size, K):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 1e6, 0.3)]
    strains = np.random.default_rng(sum(size)).uniform(-5e-3, 5e-3, (2, 6))
    r = mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, (9.0, 8.0, 0.1, 0.2), mats)
    ms = mp.MSolver(r, K)
    print(size, K, "coarse DOFs and widths", ms.coarse(False)[0].tolist(), flush=True)
    sig, ctan, stats, resid, ok = mp.homogenize_mixed(ms, strains, max_inner_its=8000)
    monkeypatch.setenv("MPPD_COARSE", "0")
    sig_j, ctan_j, stats_j, resid_j, ok_j = mp.homogenize_mixed(mp.MSolver(r, K), strains, max_inner_its=8000)
    assert ok and ok_j and resid.max() < 1e-8 and resid_j.max() < 1e-8
    assert rel(sig, sig_j) < 1e-6 and rel(ctan, ctan_j) < 1e-6
    assert stats[1] < stats_j[1]
