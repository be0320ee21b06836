"""lulesh_lagrange_leapfrog_noalloc takes the final time constraints on the host
from the partial minima its last element kernel left: fields and scalars bit
for bit those of lulesh_lagrange_leapfrog at the ends of each form's range."""
import pytest

from test_zz_no_alloc import run_both


@pytest.mark.gpu
@pytest.mark.parametrize("nx", [1, 2, 9, 31, 32, 33, 40, 41, 67])
@pytest.mark.parametrize("quirks", [7, 0])
def test_noalloc_constraints_of_every_form(nx, quirks):
    run_both(nx, 4, quirks)
