"""GPU: the multilevel preconditioner at high and low contrast, where the coarse nodes have to be nodes of its second level.

Coarse elements of 5, 3 or 4, and 4 or 5 fine ones; many small spheres, and a layer whose edge lies on a coarse node of
odd index (50 elements, at 15).  sigma within 1e-5 of the Jacobi solver's (both to 1e-8 of the start residual, times a
condition number that grows with the contrast; 1e-6 at contrast 10), with fewer inner iterations."""
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


@pytest.mark.parametrize("size, micro, contrast", [
    ((31, 31, 31), "spheres", 1e4), ((31, 31, 31), "spheres", 1e5), ((36, 35, 37), "spheres", 1e4),
    ((51, 51, 51), "layer", 1e4), ((51, 51, 51), "layer", 1e-5), ((41, 41, 41), "spheres", 1e5),
    ((33, 33, 65), "spheres", 1e4)])
def test_against_jacobi(mp, monkeypatch, size, micro, contrast):
    mats = [mp.material(0, 1e6, 0.3)] + [mp.material(0, 1e6 * contrast, 0.25)] * 2
    r = (mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, (3.0, 40.0, 0.02, 0.08), mats) if micro == "spheres" else
         mp.Rve(size, mp.MIC_LAYER_Y, (0.3, 0, 0, 0), mats))
    e = np.random.default_rng(8).uniform(-5e-3, 5e-3, (2, 6))
    sig, stats, rel, ok = mp.MSolver(r, 4).solve(e, max_inner_its=20000)
    monkeypatch.setenv("MPPD_COARSE", "0")
    sig_j, stats_j, rel_j, ok_j = mp.MSolver(r, 4).solve(e, max_inner_its=20000)
    print(size, micro, contrast, "inner iterations", stats, "Jacobi", stats_j, "sigma",
          np.abs(sig - sig_j).max() / np.abs(sig_j).max(), flush=True)
    assert ok and ok_j and np.abs(sig - sig_j).max() < 1e-5 * np.abs(sig_j).max()
    assert stats[1] < stats_j[1]


@pytest.mark.parametrize("size, contrast", [((31, 31, 31), 1e5), ((17, 14, 18), 1e6)])
def test_passes_that_end_in_jacobi(mp, monkeypatch, size, contrast):
    """More than 500 iterations a pass: solve, Newton and adjoint go on with Jacobi and converge with one outer pass
    more at most, to the same sigma (as above)."""
    mats = [mp.material(0, 1e6, 0.3)] + [mp.material(0, 1e6 * contrast, 0.25)] * 2
    r = mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, (3.0, 40.0, 0.02, 0.08), mats)
    e = np.random.default_rng(9).uniform(-5e-3, 5e-3, (2, 6))
    ms = mp.MSolver(r, 8)
    monkeypatch.setenv("MPPD_COARSE", "0")
    mj = mp.MSolver(r, 8)
    calls = []
    for m in (ms, mj):
        sig, stats, rel, ok = m.solve(e, max_inner_its=8000)
        nsig, out, nstats = m.newton(e, cg_rel_tol=1e-8, nr_rel_tol=1e-6, mixed=(1e-5, 8000, 10))
        ctan, asig, dmat, astats, arel, aok = m.adjoint(e, max_inner_its=8000)
        calls.append((sig, nsig, asig, ctan))
        print(size, contrast, stats, nstats, astats, flush=True)
        assert ok and aok and (out[:, 2] == 1).all()
    for a, b in zip(*calls):
        assert np.abs(a - b).max() < 1e-5 * np.abs(b).max()
