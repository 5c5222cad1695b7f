"""FP32 potentials of many species at the pixel counts where the tile kernel
takes over (3M pixels up to 8 species, 6M with more): a stack equals its slices
computed one at a time by the per-pixel kernel, bit for bit."""
import pytest

from test_gpu_potential_splat_tiles import test_stack_equals_single_slices as stack_equals_single_slices

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nslice,nspecies,natoms", [
    (1000, 700, 5, 8, 900), (1024, 996, 6, 9, 1200), (1024, 996, 7, 9, 1200), (1024, 996, 7, 20, 2000),
])
def test_many_species(ctx, nx, ny, nslice, nspecies, natoms):
    stack_equals_single_slices(ctx, nx, ny, nslice, 90.0, 100.0, 1.7, nspecies, natoms)
