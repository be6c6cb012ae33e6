"""GPU: elastic mixed-precision batches solved far beyond the usual tolerance, against the FP64 batch.

Both solve to 1e-12 of the start's D^-1-scaled residual.  Stresses then agree to that times the condition number of the
scaled matrix, below 1e3 at these sizes and contrast: 1e-9.  Coarse grids of 1 to 1029 DOFs, and none; a coarse node under
which up to 125 nodes are summed."""
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


@pytest.mark.parametrize("sizes", [[(5, 5, 5), (12, 14, 18), (20, 20, 20)], [(31, 29, 30), (4, 9, 9)], [(41, 41, 41)]],
                         ids=["small", "ragged", "large"])
def test_mixed_batch_equals_fp64_batch(mp, sizes):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    eps = np.random.default_rng(4).uniform(-5e-3, 5e-3, (len(sizes), 6))
    sig = []
    for mixed in (0, 1):
        b = mp.Batch([dict(size=s, micro_type=mp.MIC_CILI_FIB_Z, geo=(0.25, 0, 0, 0), materials=mats) for s in sizes],
                     lin_stress=0, nr_max_its=1, nr_rel_tol=1e-14, cg_rel_tol=1e-12, cg_max_its=4000,
                     mixed_precision=mixed)
        b.set_strains(eps)
        b.homogenize()
        sig.append(b.stress())
        if mixed:
            print(sizes, "mixed stats", b.mixed_stats(), flush=True)
    err = np.abs(sig[1] - sig[0]).max(axis=1) / np.abs(sig[0]).max(axis=1)
    print("relative difference", err, flush=True)
    assert (err <= 1e-9).all()
