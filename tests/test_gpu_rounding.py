"""Rounding of the factorisations' parts on their own: each against the same quantity
in extended precision from the same 64-bit inputs, at the precision of sums that start
from zero and are taken off once."""
import numpy as np
import pytest
import scipy.linalg

from camellia2_amd import dpg

from helpers import cdr2d, poisson2d, poisson3d, stokes2d

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

LD = np.longdouble


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def eliminate(a, n):
    """the Schur complement of a's first n rows and columns, in extended precision"""
    a = a.astype(LD)
    for j in range(n):
        a[j + 1:, j + 1:] -= np.outer(a[j + 1:, j] / a[j, j], a[j, j + 1:])
    return a[n:, n:]


# F = 12, 27, 28, 32 and 27 field columns of cells factored in LDS, 48 and 112 through the panels
@pytest.mark.parametrize("case", [poisson2d(3, 2, k=2, kt=3), poisson2d(3, 2), stokes2d(2, 1, k=2, kt=3),
                                  poisson3d(2, 1, 1, k=2, kt=2), cdr2d(2, 2), poisson2d(2, 1, k=4, kt=6),
                                  stokes2d(2, 1)], ids=["12", "27", "28", "32", "cdr", "48", "112"])
def test_schur_complement_of_its_own_K(case):
    f, b, nodes, par, coefs, load = case
    F = dpg.sizes(f, b).F
    A = dpg.LocalAssembler(f, [b])
    out, bad = A.local_stiffness_and_rhs(0, dev(nodes), dev(par), dev(coefs), load, want_schur=True)
    assert bad == 0
    A.close()
    out = {k: v.cpu().numpy() for k, v in out.items()}
    mine = lapack = 0.0
    for K, rhs, S, r in zip(out["K"], out["rhs"], out["schur"], out["schur_rhs"]):
        M = K.shape[0]
        a = np.zeros((M + 1, M + 1))
        a[:M, :M], a[M, :M], a[:M, M] = K, rhs, rhs
        T = M - F
        ref = eliminate(a, F)[:, :T]
        s = 1.0 / np.sqrt(np.diag(K)[:F])
        X = scipy.linalg.solve_triangular(np.linalg.cholesky(K[:F, :F] * s[:, None] * s), s[:, None] * a[:F, F:], lower=True)
        cpu = (a[F:, F:] - X.T @ X)[:, :T]
        mine = max(mine, float(np.linalg.norm((np.vstack([S, r]) - ref).astype(np.float64)) / np.linalg.norm(K)))
        lapack = max(lapack, float(np.linalg.norm((cpu - ref).astype(np.float64)) / np.linalg.norm(K)))
    print(f"F {F}: {mine:.2e} of |K|, LAPACK's {lapack:.2e}")
    # the same number of roundings of the same sizes in another order
    assert mine <= 2.0 * lapack
