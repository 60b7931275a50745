"""Rounding of the factorisations' parts on their own: each against the same quantity
in extended precision from the same 64-bit inputs, at the precision of sums that start
from zero and are taken off once."""
from fractions import Fraction

import numpy as np
import pytest
import scipy.linalg

from camellia2_amd import capi, dpg
from camellia2_amd.workloads import split_quads

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


def triangles(k, kt):
    f, _, nodes, par, _, load = poisson2d(2, 1)
    nodes, par = split_quads(nodes, par)
    return f, dpg.bucket(capi.TRI, k, kt), nodes, par, None, load


# F = 12, 27, 28, 32, 27 and 63 (from column 76: two blocks of columns) field columns of
# cells factored in LDS, 48 and 112 through the panels
@pytest.mark.parametrize("case", [poisson2d(3, 2, k=2, kt=3), poisson2d(3, 2), stokes2d(2, 1, k=2, kt=3),
                                  poisson3d(2, 1, 1, k=2, kt=2), cdr2d(2, 2), triangles(6, 6),
                                  poisson2d(2, 1, k=4, kt=6), stokes2d(2, 1)],
                         ids=["12", "27", "28", "32", "cdr", "63", "48", "112"])
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


# a pivot 1 - n e^2 after n columns whose products e^2 are each below half a unit of 1:
# the third and the second block of 64 columns of a field block in LDS, and the second
# half of a 128-column panel (F = 192)
@pytest.mark.parametrize("k,row,n", [(7, 146, 128), (7, 127, 64), (7, 64, 64), (8, 127, 64), (8, 64, 64), (8, 191, 128)])
def test_small_products_add_up_before_they_meet_the_pivot(k, row, n):
    f, b = dpg.form("poisson", 2), dpg.bucket(capi.QUAD, k, k + 1)
    s = dpg.sizes(f, b)
    e = np.sqrt(0.24 * 2.0 ** -54)  # four products together stay below 2^-54, half the spacing below 1
    K = np.eye(s.M)
    K[row, :n] = K[:n, row] = e
    rhs = np.zeros(s.M)
    rhs[row] = 1.0
    u = torch.zeros((1, s.M), dtype=torch.float64, device="cuda:0")
    A = dpg.LocalAssembler(f, [b])
    assert A.recover_fields(0, dev(K[None]), dev(rhs[None]), u) == 0
    A.close()
    exact = float(1 / (1 - n * LD(e) * LD(e)))
    got = u[0, row].item()
    print(f"F {s.F}, row {row}: 1 + {got - 1:.2e}, exactly 1 + {exact - 1:.2e}")
    # the sum's roundings are relative to n e^2; then the pivot, its root's reciprocal (2),
    # the product with it and the last quotient: five units of 2^-53 at most
    assert abs(got - exact) <= 5 * 2.0 ** -53


# N = 21 and 65 (a lane a dof, a second one), 133 (the substitution over LDS)
@pytest.mark.parametrize("case", [poisson2d(2, 2, k=2, kt=2), poisson2d(2, 1), poisson2d(1, 1, k=3, kt=6)],
                         ids=["21", "65", "133"])
def test_error_representation_is_the_back_substitution(case):
    """with u = 0 the residual row is the load's, whose factored columns are kept: the
    substitution with quotients and fused products, each rounded once, gives the bits"""
    f, b, nodes, par, coefs, load = case
    s = dpg.sizes(f, b)
    A = dpg.LocalAssembler(f, [b])
    out, bad = A.local_stiffness_and_rhs(0, dev(nodes), dev(par), dev(coefs), load, want_factor=True)
    assert bad == 0
    u = torch.zeros((nodes.shape[0], s.M), dtype=torch.float64, device="cuda:0")
    e = A.riesz_representation(0, dev(nodes), dev(par), u, dev(coefs), load).cpu().numpy()
    A.close()
    factor, scale = out["factor"].cpu().numpy(), out["factor_scale"].cpu().numpy()
    for c in range(min(2, nodes.shape[0])):
        L = factor[c, :s.N]
        x = factor[c, s.N + s.M].copy()
        for j in range(s.N - 1, -1, -1):
            x[j] = x[j] / L[j, j]
            for i in range(j):
                x[i] = float(Fraction(x[i]) - Fraction(L[j, i]) * Fraction(x[j]))
        assert np.array_equal(e[c], x * scale[c])
