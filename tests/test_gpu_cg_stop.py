"""The end of dpg_skeleton_solve on systems that are not positive definite: an error, and
the last iterate in x."""
import pytest

from camellia2_amd import capi

from test_gpu_cg import system

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def solve(sysm, vals, load, fixed, x0, **kw):
    """x after the solve, and whether it failed"""
    x = x0.clone()
    try:
        sysm.solve(vals, load, fixed, x, tol=1e-12, **kw)
        return x, False
    except capi.DPGError as e:
        assert "positive definite" in str(e)
        return x, True


# tens and hundreds of blocks
@pytest.mark.parametrize("shape,k", [((24, 21), 3), ((88, 77), 3)])
def test_the_last_iterate_stays(shape, k):
    sysm, vals, load, n, _ = system("poisson", shape, k)
    fixed = torch.zeros(n, dtype=torch.int32, device="cuda")
    x0 = torch.linspace(-1.0, 1.0, n, dtype=torch.float64, device="cuda")
    x, failed = solve(sysm, -vals, load, fixed, x0)  # at the first step
    assert failed and torch.equal(x, x0)
    # one negative direction, reached after some steps: two coupled unknowns, their entry
    # three times their diagonal's mean, with no load of their own
    rp, col = sysm.pattern()
    rp, col = rp.cpu(), col.cpu().long()
    where = lambda i, j: int(rp[i]) + int((col[int(rp[i]):int(rp[i + 1])] == j).nonzero()[0, 0])  # noqa: E731
    j = n - 1
    k = int(col[int(rp[j])])
    v, one = vals.clone(), load.clone()
    v[where(j, k)] = v[where(k, j)] = 3 * (v[where(j, j)] * v[where(k, k)]).sqrt()
    one[j] = one[k] = 0.0
    zero = torch.zeros_like(x0)
    steps = 0
    while not solve(sysm, v, one, fixed, zero, maxit=steps + 1)[1]:
        steps += 1
        assert steps < 200
    assert steps > 0
    x, failed = solve(sysm, v, one, fixed, zero)
    last = solve(sysm, v, one, fixed, zero, maxit=steps)[0]
    print(f"{n} unknowns: not positive definite after {steps} steps")
    assert failed and torch.equal(x, last)
