"""GPU: how many iterations the FP64 CG queues past the end of a solve.

The first chunk follows the last solve, but a short solve behind long ones pays for at most 32 iterations and one for
each long one in a row before it; a row of like solves is queued to its end at once."""
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


def calls(mp, tolerances):
    """(iterations, queued past the end) of CG solves of one system to these tolerances."""
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    r = mp.Rve((22, 23, 24), mp.MIC3D_RANDOM_SPHERES, (7.0, 8.0, 0.05, 0.15), mats)
    s, u, b, x = mp.Solver(r), mp.DeviceArray(r.nrow), mp.DeviceArray(r.nrow), mp.DeviceArray(r.nrow)
    s.set_displ_bc(np.array([1e-3, 0, 0, 2e-3, 0, 0]), u)
    s.assembly_rhs(u, None, b)
    s.assembly_mat(None)
    out, before = [], 0
    for tol in tolerances:
        its = s.cg(b, x, rel_err=tol)[0]
        queued = s.cg_queued()
        out.append((its, queued - before - its))
        before = queued
    print(out, flush=True)
    return out


@pytest.mark.parametrize("pattern", ["LS", "LLS", "LLSS", "LLLLS"])
def test_short_solves_behind_long_ones(mp, pattern):
    out = calls(mp, [1e-10 if c == "L" else 0.3 for c in pattern * 3])
    long_run = max(len(q) for q in pattern.split("S"))
    for c, (its, idle) in zip(pattern * 3, out):
        assert its > 60 if c == "L" else its < 20
        assert idle <= 32 + long_run + 1  # (a long one behind a short one is none too few either)


def test_like_solves_are_queued_at_once(mp):
    out = calls(mp, [1e-6] * 72)
    assert len({its for its, _ in out}) == 1 and 32 < out[0][0] < 96
    assert all(idle == 1 for _, idle in out[-5:])


def test_solves_that_need_no_iteration(mp):
    """A right-hand side of zero is converged at the start: the next such call queues four iterations."""
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 1e7, 0.25)]
    r = mp.Rve((12, 12, 12), mp.MIC3D_RANDOM_SPHERES, (7.0, 8.0, 0.05, 0.15), mats)
    s, b, x = mp.Solver(r), mp.DeviceArray(r.nrow), mp.DeviceArray(r.nrow)
    s.assembly_mat(None)
    queued = [0]
    for _ in range(4):
        assert s.cg(b, x)[0] == 0 and not x.numpy().any()
        queued.append(s.cg_queued())
    assert np.diff(queued).tolist() == [32, 4, 4, 4]
