"""GPU: the mixed-precision batch's inner CG at the edges of its coarse grid.

Sides of 2 to 4 elements (no coarse level, two coarse elements, one interior coarse node), sides without a divisor
(coarse elements of two widths), a side much longer than the others, and RVEs with and without a coarse level in one
batch.  Against the FP64 batch: both solve D^-1-scaled residuals to 1e-10 of their start, so displacements, and the
stresses that average them, agree to 1e-10 times the condition number of the scaled matrix, below 1e3 at these sizes
and contrast."""
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


BATCHES = {
    "none": [(3, 3, 3), (4, 4, 4), (4, 9, 9)],
    "smallest": [(5, 5, 5), (5, 6, 7), (6, 5, 12)],
    "primes": [(12, 14, 18), (20, 20, 20), (24, 12, 8)],
    "long": [(45, 5, 6), (6, 61, 5), (5, 6, 95)],
    "mixed": [(4, 4, 4), (18, 18, 18), (3, 20, 20), (11, 11, 11), (2, 2, 2)],
}


@pytest.mark.parametrize("law", ["elastic", "j2"])
@pytest.mark.parametrize("name", list(BATCHES))
def test_mixed_batch_equals_fp64_batch(mp, name, law):
    mats = [mp.material(0, 1e6, 0.3) if law == "elastic" else mp.material(1, 1e6, 0.3, 1e5, 1e4),
            mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    sizes = BATCHES[name]
    rng = np.random.default_rng(3)
    eps = rng.normal(size=(len(sizes), 6))
    eps *= 8e-3 / np.linalg.norm(eps, axis=1, keepdims=True)
    sig = []
    for mixed in (0, 1):
        b = mp.Batch([dict(size=s, micro_type=mp.MIC_CILI_FIB_Z, geo=(0.25, 0, 0, 0), materials=mats) for s in sizes],
                     lin_stress=0, nr_max_its=8, nr_rel_tol=1e-9, cg_rel_tol=1e-10, cg_max_its=2000,
                     mixed_precision=mixed)
        b.set_strains(eps)
        b.homogenize()
        sig.append(b.stress())
    scale = np.abs(sig[0]).max(axis=1, keepdims=True)
    assert (np.abs(sig[1] - sig[0]) <= 1e-7 * scale).all()
