"""GPU: displacement outputs of the multi-RHS Newton that share a vector: the last field's is what it holds."""
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


@pytest.mark.parametrize("same", [(0, 0, 0, 0, 0), (0, 1, 0, 1, 0), (0, 1, 2, 2, 1), (0, None, 0, None, 1)])
def test_shared_output_vectors(mp, same):
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    r = mp.Rve((41, 40, 39), mp.MIC_SPHERE, (0.3, 0, 0, 0), mats)
    e = np.random.default_rng(6).uniform(-5e-3, 5e-3, (5, 6))
    own = [mp.DeviceArray(r.nrow) for _ in same]
    mp.MSolver(r, 8).newton(e, u_out=own)
    vec = [mp.DeviceArray(r.nrow) for _ in range(3)]
    mp.MSolver(r, 8).newton(e, u_out=[None if k is None else vec[k] for k in same])
    for k in {k for k in same if k is not None}:
        last = max(i for i, q in enumerate(same) if q == k)
        assert np.array_equal(vec[k].numpy(), own[last].numpy())
