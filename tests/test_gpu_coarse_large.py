"""GPU: the coarse level of multi-RHS solvers on large RVEs and at high contrast.

Above 80 elements a side a coarse element is 8 or more fine ones wide; with elements of two widths h and h + 1 a fine
element has (2 h + 1)^3 positions in its coarse element, and the set-up holds them in slabs.  Above a contrast of 30 the
coarse nodes have even fine indices: up to three widths a side.  Every side up to 255
elements has a coarse level, whatever divides it."""
import numpy as np
import pytest

pytestmark = pytest.mark.gpu

GEO = (777.0, 6.0, 0.08, 0.2)
CORNER = [(0, 0, 0), (1, 0, 0), (1, 1, 0), (0, 1, 0), (0, 0, 1), (1, 0, 1), (1, 1, 1), (0, 1, 1)]


@pytest.fixture(scope="module")
def mp():
    import micropp_amd

    micropp_amd.load()
    if not micropp_amd.gpu_available():
        pytest.skip("no HIP device")
    return micropp_amd


def materials(mp, contrast=10.0):
    return [mp.material(0, 1e6, 0.3)] + [mp.material(0, 1e6 * contrast, 0.25)] * 2


@pytest.mark.parametrize("elems", [(135, 135, 135), (144, 144, 144), (120, 92, 158), (131, 40, 255)],
                         ids=lambda s: "x".join(map(str, s)))
def test_large_rves_have_a_coarse_level(mp, elems):
    r = mp.Rve([n + 1 for n in elems], mp.MIC3D_RANDOM_SPHERES, GEO, materials(mp))
    dims = mp.MSolver(r, 4).coarse(False)[0]
    print(elems, "coarse", dims.tolist(), flush=True)
    assert dims[0] > 0
    for ne, h, m in zip(elems, dims[1:4], dims[4:]):  # widths h, or h and h + 1
        assert h * (m + 1) <= ne <= (h + 1) * (m + 1)


def stiffness(mp, r, E, nu):
    lam, mu = nu * E / ((1 + nu) * (1 - 2 * nu)), E / (2 * (1 + nu))
    c = np.diag([2 * mu] * 3 + [mu] * 3)
    c[:3, :3] += lam
    return sum(b.T @ c @ b for b in r.bmat().reshape(8, 6, 24)) / (8 * r.nelem)


def side(ne, d, even):
    """Coarse element, position from its first fine element and width, of every fine element of a side."""
    if even and (ne % d or ne // d % 2):
        at = np.array([2 * (q * ((ne + 1) // 2) // d) for q in range(d)] + [ne])
    else:
        at = np.array([q * ne // d for q in range(d + 1)])
    e = np.searchsorted(at, np.arange(ne), side="right") - 1
    return e, np.arange(ne) - at[e], (at[1:] - at[:-1])[e]


# slabs of 14 of 17 planes of positions, of 5 of 27, and one slab
@pytest.mark.parametrize("elems, contrast", [((85, 83, 82), 10.0), ((131, 131, 127), 10.0), ((40, 36, 31), 10.0),
                                             ((40, 36, 31), 100.0), ((33, 35, 30), 100.0), ((85, 83, 82), 100.0)],
                         ids=str)
def test_coarse_inverse_of_slabs(mp, elems, contrast):
    """Against the inverse of the Galerkin matrix formed here from element matrices and hats; the bar of the small
    grids: 1e-6 of the largest entry (FP32 rounding of the entries is 6e-8 of each)."""
    r = mp.Rve([n + 1 for n in elems], mp.MIC3D_RANDOM_SPHERES, GEO, materials(mp, contrast))
    dims, ainv = mp.MSolver(r, 4).coarse()
    m = [int(v) for v in dims[4:]]
    d = [v + 1 for v in m]
    ke = [stiffness(mp, r, 1e6, 0.3)] + [stiffness(mp, r, 1e6 * contrast, 0.25)] * 2
    phase = r.elem_types().reshape(elems[::-1])
    sides = [side(ne, n, contrast > 30) for ne, n in zip(elems, d)]
    kinds = [sorted(set(zip(p.tolist(), w.tolist()))) for _, p, w in sides]
    sums = np.zeros((d[2] * d[1] * d[0], 24, 24))

    def line(a, kind):  # the fine elements of a kind along a side, their coarse elements, their two nodes' hats
        e, p, w = sides[a]
        at = np.flatnonzero((p == kind[0]) & (w == kind[1]))
        x = (kind[0] + np.array([0, 1])) / kind[1]
        return at, e[at], np.stack([1 - x, x], 1)

    for kz in kinds[2]:
        z, ez, wz = line(2, kz)
        for ky in kinds[1]:
            y, ey, wy = line(1, ky)
            for kx in kinds[0]:
                x, ex, wx = line(0, kx)
                n = np.array([[wx[a[0], c[0]] * wy[a[1], c[1]] * wz[a[2], c[2]] for c in CORNER] for a in CORNER])
                p = np.kron(n, np.eye(3))
                c = np.stack([p.T @ k @ p for k in ke])
                coarse = ((ez[:, None, None] * d[1] + ey[:, None]) * d[0] + ex).ravel()
                sums[coarse] += c[phase[np.ix_(z, y, x)].ravel()]
    nodes = np.array([[((ez + c[2]) * (d[1] + 1) + ey + c[1]) * (d[0] + 1) + ex + c[0] for c in CORNER]
                      for ez in range(d[2]) for ey in range(d[1]) for ex in range(d[0])])
    full = (d[0] + 1) * (d[1] + 1) * (d[2] + 1)
    k, j, i = np.meshgrid(np.arange(d[2] + 1), np.arange(d[1] + 1), np.arange(d[0] + 1), indexing="ij")
    inner = ((i > 0) & (i < d[0]) & (j > 0) & (j < d[1]) & (k > 0) & (k < d[2])).ravel()
    number = np.full(full, -1)
    number[inner] = np.arange(inner.sum())
    dof = (number[nodes][:, :, None] * 3 + np.arange(3)).reshape(len(nodes), 24)
    dof[np.repeat(number[nodes] < 0, 3, 1)] = int(dims[0])  # boundary: a row and column dropped below
    A = np.zeros((int(dims[0]) + 1,) * 2)
    for q, kc in zip(dof, sums):
        np.add.at(A, (q[:, None], q[None]), kc)
    ref = np.linalg.inv(A[:-1, :-1])
    err = np.abs(ainv.astype(np.float64) - ref).max() / np.abs(ref).max()
    print(elems, dims.tolist(), f"max error {err:.2e}", flush=True)
    assert np.array_equal(ainv, ainv.T) and err < 1e-6


def test_large_rve_against_jacobi(mp, monkeypatch):
    """sigma of a 135^3 RVE as with Jacobi alone (both to 1e-8 of the start residual: 1e-6), in fewer iterations."""
    r = mp.Rve((136, 136, 136), mp.MIC3D_RANDOM_SPHERES, GEO, materials(mp))
    e = np.random.default_rng(0).uniform(-5e-3, 5e-3, (2, 6))
    sig, stats, rel, ok = mp.MSolver(r, 4).solve(e, max_inner_its=8000)
    monkeypatch.setenv("MPPD_COARSE", "0")
    sig_j, stats_j, rel_j, ok_j = mp.MSolver(r, 4).solve(e, max_inner_its=8000)
    print("inner iterations", stats[1], "Jacobi", stats_j[1], flush=True)
    assert ok and ok_j and np.abs(sig - sig_j).max() < 1e-6 * np.abs(sig_j).max()
    assert stats[1] < stats_j[1]
