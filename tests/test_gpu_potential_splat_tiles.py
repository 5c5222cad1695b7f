"""Large FP32 potentials take a tile kernel with the radial tables in LDS; it
sums the same pairs in the same order as the per-pixel kernel that smaller
calls take, so a stack equals its slices computed one at a time, bit for bit.

Sizes: whole and ragged tiles, cutoffs of a fraction of and beyond the bins, a
cell smaller than twice the radius (every atom near a periodic image), the most
and the fewest species, atoms exactly on pixels (the clamp of small distances)
and slices without atoms.
"""
import numpy as np
import pytest

import multislice_amd as msx

pytestmark = pytest.mark.gpu
DZ = 2.0


def atoms_of(n, a, b, nslice, nspecies, pix, seed):
    rng = np.random.default_rng(seed)
    at = np.zeros(n, msx.ATOM_DTYPE)
    at["x"], at["y"] = rng.uniform(-0.1 * a, 1.1 * a, n), rng.uniform(0, b, n)
    k = rng.integers(0, nslice - 1, n)  # the last slice is empty
    at["z"] = (k + 0.5) * DZ
    at["Z"] = rng.permutation(np.arange(1, 104))[rng.integers(0, nspecies, n)]
    at["occ"] = rng.uniform(0.5, 1.0, n)
    at["x"][:3], at["y"][:3] = [0.0, 5 * pix[0], 0.0], [0.0, 7 * pix[1], 3 * pix[1]]
    return at, k


@pytest.mark.parametrize("nx,ny,nslice,a,b,radius,nspecies,natoms", [
    (512, 512, 13, 51.2, 51.2, 3.0, 3, 1500),
    (1000, 787, 5, 70.0, 60.0, 2.3, 1, 800),
    (1024, 1024, 4, 15.0, 12.0, 8.0, 5, 60),
    (1024, 996, 4, 90.0, 100.0, 0.9, 20, 2000),
    (2000, 520, 4, 140.0, 40.0, 12.0, 21, 300),
    (33, 1500, 70, 3.0, 150.0, 1.0, 2, 1000),
])
def test_stack_equals_single_slices(ctx, nx, ny, nslice, a, b, radius, nspecies, natoms):
    at, k = atoms_of(natoms, a, b, nslice, nspecies, (a / nx, b / ny), nx + ny)
    V = ctx.potential(at, (a, b, DZ * nslice), nx, ny, nslice, radius)
    assert V[0].max() > 0
    for z in range(nslice):
        one = at[k == z].copy()
        one["z"] = 0.5 * DZ
        want = ctx.potential(one, (a, b, DZ), nx, ny, 1, radius)[0]
        np.testing.assert_array_equal(V[z], want, err_msg=f"slice {z}")
