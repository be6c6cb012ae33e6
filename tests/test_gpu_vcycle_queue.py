"""GPU: inner iterations queued past the end of a solve with the multilevel preconditioner, whose iterations are long.

Chunks hold at most 16 iterations, and a solve's last one at least one of its own: at most 15 idle ones a pass, also where
the residual stays on a plateau (high contrasts) and its rate foretells hundreds."""
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


@pytest.mark.parametrize("size", [(15, 15, 15), (31, 31, 31)])
@pytest.mark.parametrize("contrast", [1e-3, 10.0, 1e3, 1e4])
@pytest.mark.parametrize("geo", [(3.0, 8.0, 0.05, 0.15), (3.0, 40.0, 0.02, 0.08)])
def test_idle_iterations(mp, size, contrast, geo):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e6 * contrast, 0.25), mp.material(0, 1e6, 0.3)]
    ms = mp.MSolver(mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, geo, mats), 8)
    e = np.random.default_rng(7).uniform(-5e-3, 5e-3, (2, 6))
    sig, ctan, stats, rel, ok = mp.homogenize_mixed(ms, e, rel_tol=1e-8, max_inner_its=8000)
    print(size, contrast, "run", stats, "queued", ms.queued(), flush=True)
    assert ok and 0 <= ms.queued() - stats[1] <= 15 * stats[0]
