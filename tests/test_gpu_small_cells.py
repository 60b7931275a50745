"""Cells whose augmented matrix is factored in LDS (D = N + M + 2 <= 192):
orders at the edges of its 16-column panels, its 64-column steps and its limit,
against the oracle under the floor rule of test_gpu_parity."""
import pytest

from helpers import cdr2d, poisson2d, poisson3d
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu


# (k, kt): N, M, D = 21, 32, 55 / 40, 32, 74 / 65, 32, 99 (one column past 64) / 65, 55, 122 /
# 96, 55, 153 (above 80 KB: one workgroup a compute unit) / 133, 55, 190 (the largest) / 133, 84, 219 (the panel kernels)
@pytest.mark.parametrize("k,kt", [(2, 2), (2, 3), (2, 4), (3, 4), (3, 5), (3, 6), (4, 6)])
def test_orders_around_the_panel_edges(k, kt):
    check_against_oracle(poisson2d(3, 2, k=k, kt=kt), want_schur=True)


def test_one_cell_hexes_and_coefficients():
    check_against_oracle(poisson3d(1, 1, 1, k=2, kt=2), want_G=True, want_schur=True)  # N 63, M 110, D 175
    check_against_oracle(cdr2d(1, 1), want_schur=True)
