"""Update tiles of cells too large for LDS: 128 counts as 64 in every output, and the
structural zeros of B are skipped at both tiles without changing a bit, at panels of
several widths."""
import pytest

from camellia2_amd import dpg

from helpers import cdr2d, poisson2d, stokes2d
from test_gpu_adjoint import dev
from test_gpu_parity import _coupled_everywhere

pytestmark = pytest.mark.gpu

torch = pytest.importorskip("torch")

# N 176, 225, 155 and 133: a last panel of 48, 97, 27 and 5 columns
CASES = [poisson2d(2, 2, k=5, kt=7), poisson2d(2, 1, k=4, kt=8), stokes2d(2, 1, k=3, kt=4), cdr2d(2, 1, k=4, kt=6)]
IDS = ["176", "225", "155", "133"]


def outputs(form, case, update):
    _, b, nodes, par, coefs, load = case
    assert dpg.sizes(form, b).N + dpg.sizes(form, b).M + 2 > 192
    A = dpg.LocalAssembler(form, [b])
    A.set_tiles(0, 64, 64, update, 0)
    o, bad = A.local_stiffness_and_rhs(0, dev(nodes), dev(par), None if coefs is None else dev(coefs), load,
                                       want_schur=True, want_G=True, want_factor=True)
    assert bad == 0
    A.close()
    return o


@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_update_tile_128_counts_as_64(case):
    one, two, three = (outputs(case[0], case, u) for u in (64, 128, 32))
    for k in one:
        assert torch.equal(one[k], two[k]) and torch.equal(one[k], three[k]), k


@pytest.mark.parametrize("update", [32, 64])
@pytest.mark.parametrize("case", CASES, ids=IDS)
def test_skipped_zeros_change_no_bit(case, update):
    one, two = (outputs(form, case, update) for form in (case[0], _coupled_everywhere(case[0])))
    for k in one:
        assert torch.equal(one[k], two[k]), k
