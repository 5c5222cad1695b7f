"""msx_potential_rec where it changes kernels: a reflection per thread below
2^19 grid points times slices, the matrix cores from there on.  The tile
edges of the matrix-core kernel (32 rows h >= 0 by 64 columns, chunks of 16
atoms, the Nyquist row and column) on grids that reach it by their number of
slices, against the oracle's FP64 coefficients, and both kernels on the same
atoms at the rule's two sides.

Tolerance as for the whole entry point: FP64 results agree to 1e-11."""
import numpy as np
import pytest

from test_gpu_potential_rec import oracle_rec, random_atoms, rel

import multislice_amd as msx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nmult,mmult,natoms,absorb,gam", [
    (16, 16, 1, 1, 1, False, 97.0), (16, 128, 1, 1, 3, True, 90.0), (64, 16, 1, 1, 4, False, 90.0),
    (128, 32, 1, 3, 17, True, 97.0), (64, 64, 3, 1, 16, False, 90.0), (32, 256, 1, 1, 33, False, 97.0),
    (256, 64, 2, 2, 5, True, 97.0), (128, 128, 1, 1, 150, True, 90.0),
])
def test_tile_edges_of_many_slices(ctx, nx, ny, nmult, mmult, natoms, absorb, gam):
    rng = np.random.default_rng(nx + 7 * ny + natoms)
    a, b, gam = 7.0, 6.0, np.deg2rad(gam)
    ns = -(-2**19 // (nx * ny))
    c = 2.0 * ns
    at = random_atoms(rng, natoms, a, b, 4.0, [8, 14])  # in the first two slices
    dw = np.where(at["Z"] == 8, 0.4, 0.3)
    ads = np.where(at["Z"] == 8, 0.05, 0.0) if absorb else np.zeros(natoms)
    Vr, Var = oracle_rec(at, a, b, c, gam, nmult, mmult, nx, ny, ns, dw, ads)
    out = ctx.potential_rec(at, (a, b, c), nx, ny, ns, dw=dw, ads=ads if absorb else None, gamma=gam, nmult=nmult,
                            mmult=mmult, prec=msx.F64, absorptive=absorb)
    V, Va = out if absorb else (out, None)
    assert rel(V, Vr) < 1e-11
    if absorb:
        assert np.linalg.norm(Va - Var) < 1e-11 * np.linalg.norm(Vr)
    # the same first slices alone: a reflection per thread
    few = ctx.potential_rec(at, (a, b, 4.0), nx, ny, 2, dw=dw, ads=ads if absorb else None, gamma=gam, nmult=nmult,
                            mmult=mmult, prec=msx.F64, absorptive=absorb)
    assert rel(few[0] if absorb else few, Vr[:2]) < 1e-11
