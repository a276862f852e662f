"""The one-launch ghost fill against the restatement's serial boundaryI, bit
for bit, ghosts of every layer included, over the ways its branches meet at
edges and corners: every axis periodic, open or walled on either side, grids
down to two cells, with and without passive scalars, single boxes and batches."""
import itertools
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from oracle.oracle import Oracle
from tests._pairs import oracle_config, random_state

pytestmark = pytest.mark.gpu
AXIS = [(3, 3), (1, 1), (2, 2), (1, 2), (2, 1)]


@pytest.mark.parametrize("grid,npas", [((2, 2, 2), 0), ((3, 2, 5), 0), ((5, 4, 3), 2)],
                         ids=["2x2x2", "3x2x5", "5x4x3-pas2"])
@pytest.mark.parametrize("precision", [_capi.GM_PRECISION_FP64, _capi.GM_PRECISION_MIXED], ids=["fp64", "mixed"])
def test_ghost_fill_all_faces(grid, npas, precision):
    print(f"case: ghost fill {grid}, {npas} passive scalars, precision {precision}, 125 boundary sets", flush=True)
    sys.stdout.flush()
    u0 = random_state(np.random.default_rng(sum(grid)), *grid, npas=npas)
    if precision == _capi.GM_PRECISION_MIXED:
        u0 = np.asfortranarray(u0.astype(np.float32).astype(np.float64))  # exact in storage
    for sides in itertools.product(AXIS, repeat=3):
        bc = sum(sides, ())
        p = _capi.make_params(*grid, 0.1, 0.1, 0.1, bc=bc, npas=npas, precision=precision)
        O = Oracle(oracle_config(p))
        O.set_u(u0)
        O.boundaryI()
        with _capi.Subdomain(p) as dev:
            dev.upload_u(u0)
            dev.boundary_u()
            np.testing.assert_array_equal(dev.download_u(), O.get_u(), err_msg=str(bc))
        O.close()
