"""GPU: the multilevel preconditioner of the multi-RHS solver.

Odd and even sides (the second level's last element 1 or 2 wide), sides below and above five coarse
elements of uneven width, sides with no common divisor, thin cells, and the smallest grids that have a
second level; three phases, a contrast of 1000 with single stiff elements (they raise the largest eigenvalue
that the smoother's damping is set from).
Bar: sigma and ctan within 1e-6 of the Jacobi-preconditioned solve (both to 1e-8 of the start residual),
with fewer inner iterations.
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


@pytest.mark.parametrize("size, geo, contrast", [
    ((5, 5, 5), (7.0, 4.0, 0.1, 0.2), 10.0), ((6, 5, 7), (8.0, 4.0, 0.1, 0.2), 10.0),
    ((10, 12, 11), (9.0, 8.0, 0.05, 0.15), 10.0), ((30, 38, 24), (10.0, 8.0, 0.05, 0.15), 10.0),
    ((17, 34, 68), (11.0, 8.0, 0.05, 0.15), 10.0), ((24, 24, 24), (12.0, 40.0, 0.02, 0.06), 1000.0),
    ((12, 40, 12), (13.0, 30.0, 0.02, 0.08), 100.0)])
def test_multilevel_against_jacobi(mp, monkeypatch, size, geo, contrast):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e6 * contrast, 0.25), mp.material(0, 1e6, 0.3)]
    strains = np.random.default_rng(sum(size)).uniform(-5e-3, 5e-3, (3, 6))
    r = mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, geo, mats)
    sig, ctan, stats, resid, ok = mp.homogenize_mixed(mp.MSolver(r, 12), strains, max_inner_its=8000)
    monkeypatch.setenv("MPPD_COARSE", "0")
    sig_j, ctan_j, stats_j, resid_j, ok_j = mp.homogenize_mixed(mp.MSolver(r, 12), strains, max_inner_its=8000)
    print(f"{size}: inner iterations {stats[1]} (Jacobi {stats_j[1]}); sigma rel {rel(sig, sig_j):.1e}", flush=True)
    assert ok and ok_j and resid.max() < 1e-8 and resid_j.max() < 1e-8
    assert rel(sig, sig_j) < 1e-6 and rel(ctan, ctan_j) < 1e-6
    assert stats[1] < stats_j[1]
