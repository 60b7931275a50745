"""The contractions at the edges of their row groups, dof chunks and point groups,
against the oracle under the floor rule of test_gpu_parity."""
import pytest

from helpers import poisson2d, poisson3d, stokes2d
from test_gpu_parity import check_against_oracle

pytestmark = pytest.mark.gpu


# B in groups of 16 (2D) or 32 (3D) trial rows, 64 rows a phase, 64 dofs of a variable a wave, 4 or 2 points at a time:
# 36 field functions (16 + 16 + 4) and exactly 64 dofs of v; 25 and 49 dofs; 8 (less than one group) and 27 in 3D
@pytest.mark.parametrize("case", [
    lambda: poisson2d(2, 1, k=6, kt=7), lambda: poisson2d(1, 2, k=5, kt=6), lambda: stokes2d(2, 2, k=2, kt=3),
    lambda: poisson3d(2, 1, 1, k=2, kt=3), lambda: poisson3d(1, 1, 1, k=3, kt=4)],
    ids=["quad k6", "quad k5", "stokes k2", "hex k2", "hex k3"])
def test_bilinear_rows_at_group_edges(case):
    check_against_oracle(case(), want_schur=True)


# G formed in place up to 80 test dofs: 21, 40 (one step of points a term), 65 (one dof past 64), 63 on a hex; 96 is past it
@pytest.mark.parametrize("case", [
    lambda: poisson2d(2, 1, k=2, kt=2), lambda: poisson2d(2, 2, k=2, kt=3), lambda: poisson2d(3, 1, k=3, kt=4),
    lambda: poisson3d(1, 1, 2, k=2, kt=2), lambda: poisson2d(1, 1, k=3, kt=5)],
    ids=["N 21", "N 40", "N 65", "hex N 63", "N 96"])
def test_gram_matrix_around_the_limit(case):
    check_against_oracle(case(), want_G=True, want_schur=True)
