"""The panels of cells too large for LDS (potrf_block and the fused panel solve)
at widths around the 16-column tiles of the diagonal block, against the oracle
under the floor rule of test_gpu_parity; and the gradient of the energy error
alone (adjoint_eta_kernel) against the general kernel, which takes the same
columns next to cotangents of zero."""
import pytest

from camellia2_amd import capi, dpg

from helpers import cdr2d, poisson2d, stokes2d
from test_gpu_adjoint import dev, rel
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# test panels of 128 columns and a last one of 48 (N 176), 97 (225), 27 (155); field panels of 75, 48 columns
# (and G's operand from 64, 81 and 25 points: whole groups of 4 and a last one of 1)
@pytest.mark.parametrize("case", [poisson2d(2, 2, k=5, kt=7), poisson2d(2, 1, k=4, kt=8), stokes2d(2, 1, k=3, kt=4)],
                         ids=["176", "225", "155"])
def test_panel_widths(case):
    check_against_oracle(case, want_schur=True)


def cdr(topology, k, kt):
    if topology == capi.QUAD:
        return cdr2d(3, 3, k=k, kt=kt)
    f, b = dpg.form("cdr", 3), dpg.bucket(topology, k, kt)
    nodes, par = dpg.mesh_hex(2, 1, 1, 0.05, 5)
    coefs = dpg.rng_uniform(6, 0.2, 1.0, 10).reshape(2, 5)
    return f, b, nodes, par, coefs, dpg.load_sine_modes(3, 1, 4, 3, 7)


# N 40 (below a wave), 65, 96, 133 (rows of L from memory), 225, and hexes of N 63 and 172
@pytest.mark.parametrize("topology,k,kt", [(capi.QUAD, 2, 3), (capi.QUAD, 3, 4), (capi.QUAD, 3, 5), (capi.QUAD, 3, 6),
                                           (capi.QUAD, 4, 8), (capi.HEX, 2, 2), (capi.HEX, 2, 3)])
def test_gradient_of_the_energy_error_alone(topology, k, kt):
    f, b, nodes, par, coefs, load = cdr(topology, k, kt)
    s = dpg.sizes(f, b)
    C = nodes.shape[0]
    A = dpg.LocalAssembler(f, [b])
    dn, dp, dc, du = dev(nodes), dev(par), dev(coefs), dev(dpg.rng_normal(11, C * s.M).reshape(C, s.M))
    zero_K = torch.zeros((C, s.M, s.M), dtype=torch.float64, device="cuda:0")
    zero_r = torch.zeros((C, s.M), dtype=torch.float64, device="cuda:0")
    out, nbad = A.local_stiffness_and_rhs(0, dn, dp, dc, load, want_factor=True)
    assert nbad == 0
    for kept in ({}, dict(factor=out["factor"], factor_scale=out["factor_scale"])):
        alone = A.adjoint(0, dn, dp, dc, load, u=du, **kept)
        general = A.adjoint(0, dn, dp, dc, load, u=du, Kbar=zero_K, rhsbar=zero_r, **kept)
        # the same factor and z: sums of up to some 1e4 terms in another order, through a
        # back substitution whose factor has a condition number below 1e4: 1e4 * 1e2 eps
        # (rounding of sums grows as the root of their length)
        e = rel(alone.cpu().numpy(), general.cpu().numpy())
        print(f"N {s.N}: the gradient alone against the general kernel {e:.2e}")
        assert e < 2.3e-10
    A.close()


# M 84 and 119: tiles of 64 and 32 with ragged last rows, the load's row at a tile's first and inner rows
@pytest.mark.parametrize("update", [32, 64])
@pytest.mark.parametrize("case", [poisson2d(2, 1, k=4, kt=7), stokes2d(2, 1, k=3, kt=4)], ids=["84", "119"])
def test_outputs_of_the_trailing_product(case, update):
    """K and rhs from the product's tiles are the same with a Schur stage behind it
    (which reads them from the workspace) and without, symmetric, and both parts of
    the Schur stage's output hold against K."""
    f, b, nodes, par, coefs, load = case
    s = dpg.sizes(f, b)
    A = dpg.LocalAssembler(f, [b])
    A.set_tiles(0, 64, 64, update)
    dn, dp, dc = dev(nodes), dev(par), dev(coefs)
    one, bad = A.local_stiffness_and_rhs(0, dn, dp, dc, load)
    two, bad2 = A.local_stiffness_and_rhs(0, dn, dp, dc, load, want_schur=True)
    assert bad == 0 and bad2 == 0
    K, rhs, F = one["K"], one["rhs"], s.F
    assert torch.equal(K, two["K"]) and torch.equal(rhs, two["rhs"])
    assert torch.equal(K, K.transpose(1, 2))
    K, rhs, S, r = (x.cpu() for x in (K, rhs, two["schur"], two["schur_rhs"]))
    assert torch.equal(S, S.transpose(1, 2))
    Z = torch.linalg.solve(K[:, :F, :F], torch.cat([K[:, :F, F:], rhs[:, :F, None]], dim=2))
    ref = torch.cat([K[:, F:, F:], rhs[:, F:, None]], dim=2) - K[:, F:, :F] @ Z
    # backward stable on both sides: the condition number of K_FF (below 1e5) times F eps
    scale = torch.linalg.matrix_norm(K[:, F:, F:]).max()
    assert (torch.cat([S, r[:, :, None]], dim=2) - ref).abs().max() < 1e5 * F * 2.3e-16 * scale
    A.close()
