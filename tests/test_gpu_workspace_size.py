"""Workspace bytes a cell: what the kernels of its path read and write, and no more for a
call than its path needs; and results that do not depend on what the workspace held."""
import numpy as np
import pytest

from camellia2_amd import capi, dpg

from helpers import cdr2d, poisson2d, poisson3d, stokes2d

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


def up(n, m):
    return -(-n // m) * m


# N + M + 2 = 74, 122 and 190 (factored in LDS), 219 and 414 (through the panels)
@pytest.mark.parametrize("case", [poisson2d(3, 2, k=2, kt=3), cdr2d(2, 2), poisson2d(2, 1, k=3, kt=6),
                                  poisson2d(2, 1, k=4, kt=6), stokes2d(2, 1)], ids=["74", "122", "190", "219", "414"])
def test_bytes_a_cell(case):
    f, b, nodes, par, coefs, load = case
    s = dpg.sizes(f, b)
    C, npr, D = nodes.shape[0], f.spatial_dim + 1, s.N + s.M + 2
    kinds = list(f.trial_kind[:f.n_trial])
    fields = sum(f.spatial_dim if k == 1 else 1 for k in kinds if k in (0, 1))
    sides = sum(k in (2, 3) for k in kinds)
    row = up(s.N, 8)
    operands = row * (f.n_ipterms * up(s.QG, 16) + fields * s.Q + sides * s.nsides * s.Qs)
    weights = npr * f.n_test * (s.QG * f.n_ipterms + s.Q * (fields + 1) + s.nsides * s.Qs * sides)
    diagonal_blocks = 64 * up(s.N + s.F, 64) if D > 192 else 0
    cell = up(D, 8) * D + operands + weights + up(max(s.N, s.M), 8) + diagonal_blocks
    A = dpg.LocalAssembler(f, [b], precision=capi.PREC_FP32)
    A.local_stiffness_and_rhs(0, dev(nodes), dev(par), dev(coefs), load, want_schur=True)
    print(f"D {D}: {A.workspace_bytes() // C} bytes a cell")
    assert A.workspace_bytes() == 8 * C * cell
    A.close()
    # the Riesz representation: the factor and its right-hand side besides where they do not lie in A
    one, two = dpg.LocalAssembler(f, [b]), dpg.LocalAssembler(f, [b])
    one.local_stiffness_and_rhs(0, dev(nodes), dev(par), dev(coefs), load, want_schur=True)
    u = torch.zeros((C, s.M), dtype=torch.float64, device="cuda:0")
    two.riesz_representation(0, dev(nodes), dev(par), u, dev(coefs), load)
    more = up((s.N + s.M + 1) * s.N, 8) + row if D <= 192 else 0
    assert two.workspace_bytes() == one.workspace_bytes() + 8 * C * more
    one.close()
    two.close()


# dense G with merged and unmerged terms' tiles of 64 and 32, sum-factorised G, cells in LDS
@pytest.mark.parametrize("case,tiles", [(poisson2d(4, 3), (64, 64, 64)), (stokes2d(3, 2), (32, 32, 32)),
                                        (stokes2d(3, 2), (64, 64, 128)), (poisson3d(2, 2, 1, k=3, kt=4), (64, 64, 32)),
                                        (poisson3d(2, 2, 1, k=3, kt=4), (32, 32, 64, 1)), (cdr2d(3, 3), (64, 64, 64))],
                         ids=["p2d", "stokes-32", "stokes-64", "p3d", "p3d-sf", "cdr"])
@pytest.mark.parametrize("precision", [capi.PREC_FP64, capi.PREC_FP32, capi.PREC_INT8SPLIT])
def test_results_do_not_depend_on_the_workspace_before(case, tiles, precision):
    """every call once on a new plan and once on one whose workspace an assembly of cells
    with NaN vertices has filled, in batches of two cells"""
    f, b, nodes, par, coefs, load = case
    s = dpg.sizes(f, b)
    dn, dp, dc = dev(nodes), dev(par), dev(coefs)
    C = nodes.shape[0]
    u = dev(dpg.rng_normal(5, C * s.M).reshape(C, s.M))
    nan = torch.full_like(dn, float("nan"))

    def results(used):
        A = dpg.LocalAssembler(f, [b], precision=precision, max_batch_cells=2)
        A.set_tiles(0, *tiles) if precision == capi.PREC_FP64 else None
        got = []

        def call(run):
            if used:
                A.local_stiffness_and_rhs(0, nan, dp, dc, load, want_schur=True)
            got.append(run())

        call(lambda: A.local_stiffness_and_rhs(0, dn, dp, dc, load, want_schur=True)[0])
        call(lambda: {"eta2": A.energy_error(0, dn, dp, u, dc, load)})
        if precision != capi.PREC_INT8SPLIT:
            call(lambda: A.local_stiffness_and_rhs(0, dn, dp, dc, load, want_G=True, want_factor=True)[0])
        if precision == capi.PREC_FP64:
            call(lambda: {"e": A.riesz_representation(0, dn, dp, u, dc, load)})
        if precision == capi.PREC_FP64 and dc is not None:
            call(lambda: dict(zip(("eta2", "grad"), A.adjoint(0, dn, dp, dc, load, u=u, want_eta2=True))))
        first = got[0]

        def fields():
            v = u.clone()
            assert A.recover_fields(0, first["K"], first["rhs"], v) == 0
            return {"u": v}

        call(fields)
        A.close()
        return got

    for new, old in zip(results(False), results(True)):
        for k in new:
            assert torch.isfinite(new[k]).all() and torch.equal(new[k], old[k]), k
