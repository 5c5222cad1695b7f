"""msx_potential_rec at the edges of its work-group tiles (32 rows h >= 0 by
64 columns, chunks of 16 atoms, 4 atoms per matrix instruction) against the
oracle's FP64 coefficients: grids smaller than a tile, the Nyquist row and
column, remainders of the atom chunks, with and without absorption factors.

Tolerance: a coefficient sums at most a few dozen unit phases whose arguments
are rounded to 2^-53 of a turn, and the FP64 transforms add about 1e-15 per
stage, so FP64 results agree to well below 1e-11.
"""
import numpy as np
import pytest

from test_gpu_potential_rec import oracle_rec, random_atoms, rel

import multislice_amd as msx

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("nx,ny,nmult,mmult,natoms,absorb", [
    (16, 16, 1, 1, 1, False), (16, 128, 1, 1, 3, True), (64, 16, 1, 1, 4, False), (128, 32, 1, 3, 17, True),
    (64, 64, 3, 1, 16, False), (32, 256, 1, 1, 33, False), (256, 64, 2, 2, 5, True),
])
def test_tile_edges(ctx, nx, ny, nmult, mmult, natoms, absorb):
    rng = np.random.default_rng(nx + 7 * ny + natoms)
    a, b, c, gam = 7.0, 6.0, 4.0, np.deg2rad(97.0)
    at = random_atoms(rng, natoms, a, b, c, [8])
    dw = np.full(natoms, 0.4)
    ads = rng.choice([0.0, 0.05], natoms) if absorb else np.zeros(natoms)
    Vr, Var = oracle_rec(at, a, b, c, gam, nmult, mmult, nx, ny, 2, dw, ads)
    out = ctx.potential_rec(at, (a, b, c), nx, ny, 2, dw=dw, ads=ads if absorb else None, gamma=gam, nmult=nmult,
                            mmult=mmult, prec=msx.F64, absorptive=absorb)
    V, Va = out if absorb else (out, None)
    assert rel(V, Vr) < 1e-11
    if absorb:
        assert np.linalg.norm(Va - Var) < 1e-11 * np.linalg.norm(Vr)
