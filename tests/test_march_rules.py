"""Which calls the marching loops take (host code only)."""
import pytest

from seistorch_amd.equations2d import acoustic_habc as ah


# few shots of large grids march; many shots of grids that are mostly frame do not
@pytest.mark.parametrize("B,nz,nx,march", [
    (1, 3000, 3000, True), (3, 2500, 2500, True), (16, 900, 2500, True), (4, 1800, 1700, True),
    (64, 450, 450, False), (500, 164, 164, False), (1, 164, 164, False), (10 ** 6, 110, 900, False)])
def test_habc_marches_by_the_cells_away_from_the_edges(B, nz, nx, march):
    assert ah._march_fits(B, nz, nx) is march
