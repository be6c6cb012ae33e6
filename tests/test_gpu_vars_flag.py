"""GPU: the history pass' nonlinear flag, from one Gauss point of any wave and from all of them at once.

The pass moves the same bytes whether the points yield or not, so its time may not hang on how many set the flag: at
most twice that of a pass in which none does (1.1 times measured, 6 times with an atomic operation a wave)."""
import time

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


def _solver(mp, size, law):
    mats = [mp.material(1, 1e6, 0.3, 1e5, 1e4) if law == "j2" else mp.material(2, 1e6, 0.3, 0.0, 0.0, 1e5)]
    r = mp.Rve(size, mp.MIC_SPHERE, (0.0, 0.0, 0.0, 0.0), mats * 3)
    return r, mp.Solver(r)


@pytest.mark.parametrize("law", ["j2", "damage"])
@pytest.mark.parametrize("size", [(2, 2, 2), (4, 4, 4), (6, 7, 8), (34, 2, 2)])
def test_one_corner_sets_the_flag(mp, size, law):
    r, s = _solver(mp, size, law)
    v = mp.DeviceArray(r.nvars)
    n = r.nrow // 3
    assert s.vars_new(mp.DeviceArray(r.nrow), None, v) == 0
    for node in (0, size[0] - 1, n - size[0], n - 1):  # corners: one element each
        u = np.zeros(r.nrow)
        u[3 * node:3 * node + 3] = 0.3, 0.2, -0.25
        assert s.vars_new(mp.DeviceArray.from_numpy(u), None, v) == 1, node
        assert s.vars_new(mp.DeviceArray(r.nrow), None, v) == 0


def test_time_does_not_depend_on_how_many_points_yield(mp):
    r, s = _solver(mp, (71, 71, 71), "j2")
    v = mp.DeviceArray(r.nvars)
    best = []
    for scale, flag in ((1e-12, 0), (1e-3, 1)):
        u = mp.DeviceArray.from_numpy(scale * np.random.default_rng(0).normal(size=r.nrow))
        t = []
        for _ in range(20):
            t0 = time.perf_counter()
            assert s.vars_new(u, None, v) == flag
            t.append(time.perf_counter() - t0)
        best.append(min(t))
    print(f"none {1e6 * best[0]:.0f} us, all {1e6 * best[1]:.0f} us", flush=True)
    assert best[1] <= 2 * best[0]
