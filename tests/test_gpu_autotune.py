"""dpg_plan_autotune chooses among tiles that the bucket's kernels take; where none does
the tile stays 64."""
import numpy as np
import pytest

from camellia2_amd import capi, dpg

from helpers import cdr2d, poisson2d, stokes2d

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")


def dev(a):
    return None if a is None else torch.from_numpy(np.ascontiguousarray(a)).to("cuda:0")


# G formed in LDS and the cells factored there (N 65, D 122); G from its operand, the
# cells in LDS (N 133, D 190); panels (N 228, D 414)
@pytest.mark.parametrize("case,precision,free",
                         [(cdr2d(3, 3), capi.PREC_FP64, ()), (poisson2d(3, 3, k=3, kt=6), capi.PREC_FP64, (0,)),
                          (poisson2d(3, 3, k=3, kt=6), capi.PREC_FP32, ()), (stokes2d(3, 2), capi.PREC_FP64, (0, 2)),
                          (stokes2d(3, 2), capi.PREC_BF16X3, (2,)), (stokes2d(3, 2), capi.PREC_INT8SPLIT, (2,))],
                         ids=["lds", "operand", "fp32", "panels", "bf16x3", "int8"])
def test_roles_without_a_tile_keep_64(case, precision, free):
    f, b, nodes, par, coefs, load = case
    A = dpg.LocalAssembler(f, [b], precision=precision)
    args = (dev(nodes), dev(par), dev(coefs), load)
    for _ in range(12):  # a trial of two equal runs keeps either one
        t = A.autotune(0, *args, sample=nodes.shape[0])
        assert all(t[r] == 64 for r in range(3) if r not in free), t
        assert all(t[r] in (32, 64) for r in free), t
    A.close()
