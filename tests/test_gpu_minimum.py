"""The launch-wide minimum (one slot per 64 workgroups, published by the last
workgroup) on grids of 2 to 130 workgroups: one below, at and above the slot
count and twice it, a single workgroup, and a tile with lanes past the plane.
get_timestep's minimum of the state and of the state after each of three steps
(the step's own reduction, whose working space the launch before left) equals
the restatement's, bit for bit, as does the state."""
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from oracle.oracle import Oracle
from tests._pairs import oracle_config, random_state

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("grid", [(2, 2, 2), (16, 16, 63), (16, 16, 64), (16, 16, 65), (16, 17, 65), (8, 8, 130)],
                         ids=lambda g: "x".join(map(str, g)))
@pytest.mark.parametrize("flux_cd", [True, False], ids=["folded", "own-pass"])
def test_minimum_over_workgroups(grid, flux_cd):
    nx, ny, nz = grid
    print(f"case: minimum over workgroups, {nx}x{ny}x{nz}, flux-CD {flux_cd}, 3 steps", flush=True)
    sys.stdout.flush()
    u0 = random_state(np.random.default_rng(nx + 7 * ny + 31 * nz), nx, ny, nz)
    p = _capi.make_params(nx, ny, nz, 1.0 / nx, 1.0 / ny, 1.0 / nz, bc=(1,) * 6, enable_flux_cd=flux_cd)
    O = Oracle(oracle_config(p))
    O.set_u(u0)
    O.boundaryI()
    O.calcprim_u()
    with _capi.Subdomain(p) as dev:
        dev.upload_u(u0)
        for _ in range(3):
            dtp = dev.cfl_dtp()
            assert dtp == O.cfl_dtp()
            dev.tstep(0.1 * dtp)
            O.tstep(0.1 * dtp)
        assert dev.cfl_dtp() == O.cfl_dtp()
        np.testing.assert_array_equal(dev.download_u(), O.get_u())
    O.close()
