"""GPU: the FP64 Jacobi-CG at the edges of its kernels.

step1 forms p and Ap of 256 rows in one kernel: its LDS runs are one per z plane up to 88 nodes a line and nine
beyond; for an uploaded matrix p is formed ahead of it.  Every form does the oracle's
arithmetic except for the order of the inner products, so a solve to 1e-6 stops within an iteration of it and
agrees to ten times that; the forms among each other differ in nothing, so they agree bit for bit."""
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


# lines of 41 nodes (staged ahead) and 42, of 87, 88 and 89, fewer rows than a block, whole blocks and a remainder
SIZES = [(2, 2, 2), (3, 3, 2), (5, 4, 6), (41, 5, 6), (42, 5, 6), (87, 3, 4), (88, 4, 3), (89, 3, 4), (17, 30, 9), (32, 16, 8), (23, 31, 50)]


@pytest.mark.parametrize("size", SIZES, ids=lambda s: "x".join(map(str, s)))
def test_solve_by_computed_and_by_uploaded_columns(mp, oracle, size):
    """An assembled matrix against the same values uploaded, and both against the oracle: chunks of 32 iterations
    end inside the solve (40 of them), so the scalars pass through the state read by the host too."""
    r = mp.Rve(size, mp.MIC3D_RANDOM_SPHERES, (7.0, 5.0, 0.1, 0.3), [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25),
                                                                   mp.material(0, 1e7, 0.25)])
    s, up = mp.Solver(r), mp.Solver(r)
    u, b = mp.DeviceArray(r.nrow), mp.DeviceArray(r.nrow)
    s.set_displ_bc([5e-3, -1e-3, 2e-3, 1e-3, 0.0, -2e-3], u)
    s.assembly_mat(u)
    s.assembly_rhs(u, None, b)
    cols, vals = s.ell()
    up.upload_vals(vals)
    x, xu = mp.DeviceArray(r.nrow), mp.DeviceArray(r.nrow)
    its, err = s.cg(b, x, 1e-50, 1e-300, 40)
    its_u, err_u = up.cg(b, xu, 1e-50, 1e-300, 40)
    assert (its, err) == (its_u, err_u) or (np.isnan(err) and np.isnan(err_u))
    assert np.array_equal(x.numpy(), xu.numpy(), equal_nan=True)
    if min(size) > 2:  # an interior: the solution is not zero
        xo, io, _ = oracle.ell_cg(r.nrow // 3, 3, 81, 13, cols, vals, b.numpy(), 1e-50, 1e-6, 40)
        it6, _ = s.cg(b, x, 1e-50, 1e-6, 40)
        assert abs(it6 - io) <= 1 and np.abs(x.numpy() - xo).max() <= 1e-5 * np.abs(xo).max()


@pytest.mark.parametrize("size", [(20, 20, 20), (21, 20, 19), (90, 10, 9), (47, 46, 45), (256, 25, 15), (257, 25, 15)],
                         ids=lambda s: "x".join(map(str, s)))
def test_stencil_table_of_elastic_rves(mp, size):
    """From 8000 nodes on (20^3; 7980 stay below) an all-elastic RVE's CG reads a stencil table instead of the
    matrix, from 1100 row blocks on (47x46x45) with a thread per node unless a line has more than 256; three phases.  Solved bit for bit as the uploaded matrix, alone and beside a J2 RVE in a batch, whose
    Newton then needs what a batch of the elastic RVE alone needs."""
    mats = [mp.material(0, 1e6, 0.3), mp.material(0, 1e7, 0.25), mp.material(0, 3e6, 0.2)]
    geo = (0.3, 0.15, 0.0, 0.0)
    for micro in (mp.MIC3D_RANDOM_SPHERES, mp.MIC_SPHERE):
        r = mp.Rve(size, micro, (7.0, 5.0, 0.1, 0.3) if micro == mp.MIC3D_RANDOM_SPHERES else geo, mats)
        s, up = mp.Solver(r), mp.Solver(r)
        u, b, x, xu = (mp.DeviceArray(r.nrow) for _ in range(4))
        s.set_displ_bc([5e-3, -1e-3, 2e-3, 1e-3, 0.0, -2e-3], u)
        s.assembly_mat(u)
        s.assembly_rhs(u, None, b)
        up.upload_vals(s.ell()[1])
        assert s.cg(b, x, 1e-50, 1e-8, 500) == up.cg(b, xu, 1e-50, 1e-8, 500)
        assert np.array_equal(x.numpy(), xu.numpy())
    j2 = [mp.material(1, 1e6, 0.3, 1e5, 1e4)] + mats[1:]
    desc = [dict(size=size, micro_type=mp.MIC_SPHERE, geo=geo, materials=m) for m in (mats, mats, j2)]
    eps = np.array([[5e-3, -1e-3, 2e-3, 1e-3, 0.0, -2e-3]] * 3)
    sig = []
    for d in (desc, desc[:1], desc[2:]):
        bt = mp.Batch(d, lin_stress=0, cg_rel_tol=1e-8, cg_max_its=1000)
        bt.set_strains(eps[:len(d)])
        bt.homogenize()
        sig.append(bt.stress())
    assert np.array_equal(sig[0][0], sig[0][1]) and np.array_equal(sig[0][0], sig[1][0])
    assert np.array_equal(sig[0][2], sig[2][0])
