"""dpg_skeleton_solve's conjugate gradients at the edges of their 256-row blocks,
64-entry row chunks and 262,144-row stride, on well conditioned blocks, checked by
the residual computed on the host."""
import numpy as np
import pytest

from camellia2_amd import capi, dpg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def system(form, shape, k):
    """a mesh's condensed system with cell blocks I + V V^T / 4, V (T, 2) of entries below 1 / sqrt(T)"""
    f = dpg.form("poisson", len(shape))
    b = dpg.bucket(capi.HEX if len(shape) == 3 else capi.QUAD, k, k + 1)
    nodes, _ = (dpg.mesh_hex if len(shape) == 3 else dpg.mesh_quad)(*shape, 0.0, 1)
    gdof, n = dpg.skeleton_numbering(f, b, dpg.vertex_ids(nodes))
    C, T = gdof.shape
    g = torch.Generator(device="cuda").manual_seed(5)
    V = (2 * torch.rand((C, T, 2), generator=g, device="cuda", dtype=torch.float64) - 1) / T ** 0.5
    S = V @ V.transpose(1, 2).contiguous() / 4 + torch.eye(T, device="cuda", dtype=torch.float64)
    sysm = dpg.CondensedSystem(gdof, n)
    ent, nent = dpg.skeleton_entities(f, b, dpg.vertex_ids(nodes), n)
    rhs = 2 * torch.rand((C, T), generator=g, device="cuda", dtype=torch.float64) - 1
    vals, load = sysm.assemble(S.contiguous(), rhs)
    return sysm, vals, load, n, (ent, nent)


def residual(sysm, vals, load, fixed, x):
    rp, col = sysm.pattern()
    A = torch.sparse_csr_tensor(rp.cpu(), col.cpu().long(), vals.cpu(), size=(sysm.nglobal, sysm.nglobal))
    r = load.cpu() - (A @ x.cpu()[:, None])[:, 0]
    r[fixed.cpu() != 0] = 0.0
    return float(r.norm())


# 16 unknowns (part of one block), 347 and 369 (two, ragged), 569 and 1561 with rows of more than 64 entries, 459,543,
# and 8 million entries in long rows (the matrix in a launch of its own)
@pytest.mark.parametrize("shape,k", [((1, 1), 2), ((7, 6), 2), ((11, 4), 2), ((5, 4), 6), ((3, 2, 2), 4),
                                     ((175, 174), 4), ((9, 9, 8), 3)])
@pytest.mark.parametrize("blocks", [False, True])
def test_converged_solutions_have_the_residual_reported(shape, k, blocks):
    sysm, vals, load, n, (ent, nent) = system("poisson", shape, k)
    if blocks:
        sysm.set_blocks(ent, nent)
    fixed = torch.zeros(n, dtype=torch.int32, device="cuda")
    fixed[::7] = 1
    x = torch.linspace(-1.0, 1.0, n, dtype=torch.float64, device="cuda")
    x0 = x.clone()
    start = residual(sysm, vals, load, fixed, x)
    it, rel = sysm.solve(vals, load, fixed, x, tol=1e-12)
    print(n, it, rel)
    assert 0 < it < 200 and rel <= 1e-12
    # the recurrence's residual and the true one differ by rounding, well below 1e-13 of the start here
    assert residual(sysm, vals, load, fixed, x) <= 1.2e-12 * start
    assert torch.equal(x[fixed != 0], x0[fixed != 0])
    # a cut-off run stops where it is told to, with the same iterates
    y, z = x0.clone(), x0.clone()
    assert sysm.solve(vals, load, fixed, y, tol=1e-12, maxit=3)[0] == min(3, it)
    assert sysm.solve(vals, load, fixed, z, tol=1e-12, maxit=3)[0] == min(3, it) and torch.equal(y, z)
    assert sysm.solve(vals, load, fixed, y, tol=1e-12, maxit=0)[0] == 0 and torch.equal(y, z)


def test_nothing_to_solve_and_indefinite_systems():
    sysm, vals, load, n, _ = system("poisson", (3, 2), 2)
    fixed = torch.zeros(n, dtype=torch.int32, device="cuda")
    x = torch.zeros(n, dtype=torch.float64, device="cuda")
    assert sysm.solve(vals, torch.zeros_like(load), fixed, x) == (0, 0.0)
    with pytest.raises(capi.DPGError):
        sysm.solve(-vals, load, fixed, x)
