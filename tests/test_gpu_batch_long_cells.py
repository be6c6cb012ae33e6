"""GPU: the mixed-precision batch's coarse level on boxes whose cells are several times as long as wide.

There the inner CG takes, to 1e-5 in 64 bits on the CPU (the same tangent, a layer, contrast 10; Jacobi alone / coarse
elements counted alike on every side / of one length on every side): 78 / 70 / 36 iterations on 5 x 29 x 29 elements,
81 / 65 / 45 on 32 x 8 x 8 and 110 / 92 / 24 on 44 x 4 x 5.  A coarse element on each side must thus leave at most 0.68
of Jacobi's iterations, the middle between 0.90, 0.80, 0.84 and 0.46, 0.56, 0.22 for the two nearest."""
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


def _run(mp, size, law):
    mats = [mp.material(0, 1e6, 0.3) if law == "elastic" else mp.material(1, 1e6, 0.3, 1e5, 1e4),
            mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    b = mp.Batch([dict(size=size, micro_type=mp.MIC_LAYER_Y, geo=(0.3, 0, 0, 0), materials=mats)], lin_stress=0,
                 nr_max_its=3, nr_rel_tol=1e-6, cg_rel_tol=1e-8, cg_max_its=3000, mixed_precision=1)
    b.set_strains(np.array([[1e-3, -5e-4, 2e-3, 2e-4, 0.0, 3e-4]]))
    b.homogenize()
    return b.stress().copy(), b.stats()[0], b.mixed_stats()


@pytest.mark.parametrize("law", ["elastic", "j2"])
@pytest.mark.parametrize("size", [(6, 30, 30), (33, 9, 9), (45, 5, 6)])
def test_long_cells_take_fewer_iterations_than_jacobi(mp, size, law, monkeypatch):
    sig, its, stats = _run(mp, size, law)
    monkeypatch.setenv("MPPD_COARSE", "0")
    ref, jacobi, _ = _run(mp, size, law)
    assert np.abs(sig - ref).max() <= 1e-5 * np.abs(ref).max()
    assert stats[1] == 0 and its <= 0.68 * jacobi
