"""GPU: the multilevel preconditioner where it has a second level, and on large grids.

The smallest grids above the two-level form with even and odd sides, single stiff elements at a contrast of 1000, thin
cells (long ones, which have two levels: test_gpu_vcycle_long_cells.py), uneven coarse elements, and sides of more than 68 nodes; the solver's damping
tells which form it took (a second level has one below 1).
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


@pytest.mark.parametrize("size, geo, contrast", [
    ((29, 29, 29), (12.0, 60.0, 0.01, 0.04), 1000.0), ((30, 29, 31), (12.0, 60.0, 0.01, 0.04), 1000.0),
    ((30, 30, 30), (9.0, 8.0, 0.05, 0.15), 10.0), ((61, 62, 26), (13.0, 30.0, 0.02, 0.08), 100.0),
    ((40, 90, 91), (14.0, 8.0, 0.05, 0.2), 10.0), ((40, 71, 26), (15.0, 8.0, 0.05, 0.15), 10.0),
    ((83, 80, 85), (16.0, 8.0, 0.05, 0.15), 10.0), ((101, 101, 101), (17.0, 60.0, 0.005, 0.02), 100.0)])
def test_three_levels_against_jacobi(mp, monkeypatch, size, geo, contrast):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e6 * contrast, 0.25), mp.material(0, 1e6, 0.3)]
    strains = np.random.default_rng(sum(size)).uniform(-5e-3, 5e-3, (2, 6))
    r = mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, geo, mats)
    ms = mp.MSolver(r, 8)
    assert 0 < ms.damping()[1] < 1
    sig, ctan, stats, resid, ok = mp.homogenize_mixed(ms, strains, max_inner_its=8000)
    monkeypatch.setenv("MPPD_COARSE", "0")
    sig_j, ctan_j, stats_j, resid_j, ok_j = mp.homogenize_mixed(mp.MSolver(r, 8), strains, max_inner_its=8000)
    print(f"{size}: inner iterations {stats[1]} (Jacobi {stats_j[1]}); sigma rel {rel(sig, sig_j):.1e}", flush=True)
    assert ok and ok_j and resid.max() < 1e-8 and resid_j.max() < 1e-8
    assert rel(sig, sig_j) < 1e-6 and rel(ctan, ctan_j) < 1e-6
    assert stats[1] < stats_j[1]
