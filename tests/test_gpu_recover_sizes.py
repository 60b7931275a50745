"""Field recovery at the edges of its 16-column panels, of a wave's 64 entries and
of the size that fits LDS (F + 1 <= 192), against a dense solve."""
import numpy as np
import pytest

from camellia2_amd import capi, dpg

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


# F = 12, 27, 48, 75, 108, 147 and 192 (the panel kernels)
@pytest.mark.parametrize("k", [2, 3, 4, 5, 6, 7, 8])
@pytest.mark.parametrize("C", [1, 5])
def test_recovered_fields_solve_the_field_block(k, C):
    f, b = dpg.form("poisson", 2), dpg.bucket(capi.QUAD, k, k + 1)
    s = dpg.sizes(f, b)
    g = torch.Generator().manual_seed(7 * k + C)
    X = torch.randn((C, s.M, s.M), generator=g, dtype=torch.float64) / np.sqrt(s.M)
    d = torch.exp(torch.randn((C, s.M, 1), generator=g, dtype=torch.float64))
    K = d * (X + X.transpose(1, 2) + 4 * torch.eye(s.M, dtype=torch.float64)) * d.transpose(1, 2)
    K = 0.5 * (K + K.transpose(1, 2))
    rhs = torch.randn((C, s.M), generator=g, dtype=torch.float64)
    u = torch.randn((C, s.M), generator=g, dtype=torch.float64)
    A = dpg.LocalAssembler(f, [b])
    got = u.clone().cuda()
    assert A.recover_fields(0, K.cuda(), rhs.cuda(), got) == 0
    got = got.cpu()
    F = s.F
    ref = torch.linalg.solve(K[:, :F, :F], (rhs[:, :F, None] - K[:, :F, F:] @ u[:, F:, None]))[:, :, 0]
    assert torch.equal(got[:, F:], u[:, F:])
    # S K_FF S has a condition number below 1e2 (its spectrum is that of 4 I plus a
    # semicircle of radius 2 sqrt 2, rescaled): F eps times it, for both solves
    err = ((got[:, :F] - ref) / d[:, :F, 0].reciprocal()).norm() / (ref / d[:, :F, 0].reciprocal()).norm()
    assert err < 2 * 1e2 * F * 2.3e-16
    K[-1, F // 2, F // 2] = -1.0  # a failing cell is reported, the others are not touched by it
    got2 = u.clone().cuda()
    assert A.recover_fields(0, K.cuda(), rhs.cuda(), got2) == 1
    if C > 1:
        assert torch.equal(got2[:-1].cpu(), got[:-1])
    A.close()
