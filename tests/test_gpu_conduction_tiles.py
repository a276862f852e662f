"""The conduction sub-step kernel (32 x 8 tiles marched along z, fluxes
exchanged between lanes) against the C restatement where its tiles and marches
end: grids one below, at and above a tile, single-plane remainders, two cells;
one, two and many sub-steps, so the result comes from each of its buffers;
every boundary kind, whose edge copies it writes itself; passive scalars; and
after a boundary hook.

E agrees to relative 1e-13: t^2.5 is within 0.501 units in the last place on the
device and 1 on the host, and the other operations round alike, so a flux
differs by a few 2^-53 of itself, and a sub-step moves E by no more than E."""
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from oracle.oracle import Oracle
from tests._pairs import oracle_config
from tests.test_gpu_conduction import BSC, TEMPSC
from tests.test_gpu_hooks import JET

pytestmark = pytest.mark.gpu


def _contact(rng, shape, npas):
    shape = tuple(m + 4 for m in shape)
    u = np.zeros((8 + npas,) + shape, order="F")
    u[0] = rng.uniform(0.5, 2.0, shape)
    u[4] = 1.5 * (1.0e6 / TEMPSC) + 0.125
    u[5] = 0.5
    u[8:] = u[0] * rng.uniform(0.1, 0.9, (npas,) + shape)
    return u


CASES = [
    # grid, kind, saturation, bc, dt factor (in conduction timesteps), passive scalars, hook
    ((2, 2, 2), 1, False, (3,) * 6, 0.5, 0, False),
    ((31, 7, 3), 1, True, (1,) * 6, 0.5, 0, False),
    ((32, 8, 5), 2, True, (3, 3, 1, 1, 2, 2), 3.0, 0, False),
    ((33, 9, 4), 2, False, (2, 1, 3, 3, 1, 2), 3.0, 0, False),
    ((33, 17, 9), 1, True, (3,) * 6, 8.0, 2, False),
    ((64, 5, 33), 2, True, (3,) * 6, 8.0, 1, False),
    ((34, 10, 6), 1, False, (1, 1, 3, 3, 3, 3), 3.0, 0, True),
]


@pytest.mark.parametrize("case", CASES, ids=["x".join(map(str, c[0])) + ("-mhd" if c[1] == 2 else "") for c in CASES])
def test_conduction_tiles(case):
    grid, kind, sat, bc, fac, npas, hook = case
    print(f"case: conduction tiles {grid}, kind {kind}, saturation {sat}, {fac} conduction timesteps, hook {hook}",
          flush=True)
    sys.stdout.flush()
    u0 = _contact(np.random.default_rng(sum(grid)), grid, npas)
    h = 1.0 / max(grid)
    p = _capi.make_params(*grid, h, h, h, bc=bc, npas=npas)
    O = Oracle(oracle_config(p, user_bc=hook))
    O.set_conduction(kind, sat, tempsc=TEMPSC, bsc=BSC)
    O.set_u(u0)
    O.boundaryI()
    O.calcprim_u()
    with _capi.Subdomain(p) as dev:
        if hook:
            dev.set_user_bc(*JET)
        dev.set_conduction(kind, sat, tempsc=TEMPSC, bsc=BSC)
        dev.upload_u(u0)
        dev.boundary_u()
        np.testing.assert_array_equal(dev.download_u(), O.get_u())
        dt = fac * O.dt_cond()
        O.tstep(dt)
        dev.tstep(dt)
        ud, uo = dev.download_u(), O.get_u()
    O.close()
    for q in [0, 1, 2, 3, 5, 6, 7] + list(range(8, 8 + npas)):
        np.testing.assert_array_equal(ud[q], uo[q], err_msg=f"field {q}")
    np.testing.assert_allclose(ud[4], uo[4], rtol=1e-13, atol=0)
    inner = (slice(2, -2),) * 3
    assert np.abs(ud[4][inner] - u0[4][inner]).max() > 1e-6 * np.abs(u0[4]).max()
