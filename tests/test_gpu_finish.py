"""The pass after the corrector (the viscous result, cooling, and the next
timestep's minimum in one) at workgroup edges: 105, 256, 512 and 544 cells of
256 a workgroup.  The minimum it reduces equals the reduction's own pass over
what it stored, bit for bit; the fields that cooling does not touch equal the
restatement's viscous step, bit for bit, and E too where the gas is too cold to
cool; E and the neutral density of a cooled gas agree to relative 1e-10, the
tolerance of the cooling tests (exp, log and pow differ between host and device)."""
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from oracle.oracle import Oracle
from tests._pairs import oracle_config, random_state

pytestmark = pytest.mark.gpu

TAB = np.array([[4.0 + 0.1 * i, -22.0 + 0.01 * i] for i in range(41)])
TAB = np.asfortranarray((10.0 ** TAB).T)


@pytest.mark.parametrize("eta", [0.0, 0.03])
@pytest.mark.parametrize("kind", ["cold-table", "table", "h-rate"])
@pytest.mark.parametrize("grid", [(5, 7, 3), (4, 8, 8), (16, 16, 2), (17, 16, 2)], ids=lambda g: "x".join(map(str, g)))
def test_finish_pass(grid, kind, eta):
    print(f"case: finish pass {grid}, {kind}, eta {eta}, 2 steps", flush=True)
    sys.stdout.flush()
    npas = 1 if kind == "h-rate" else 0
    tempsc = {"cold-table": 1.0e2, "table": 1.0e6, "h-rate": 1.0e4}[kind]
    ck = _capi.GM_COOL_H if kind == "h-rate" else _capi.GM_COOL_DMC
    tab = None if kind == "h-rate" else TAB
    psc, tsc = (1.0, 1.0e13) if kind == "h-rate" else (1e-22, 10.0)
    u0 = random_state(np.random.default_rng(sum(grid)), *grid, npas=npas, vmax=0.3, bmax=0.3)
    p = _capi.make_params(*grid, 0.1, 0.1, 0.1, bc=(3, 3, 1, 1, 2, 2), npas=npas, eta=eta)
    eos = (_capi.GM_EOS_H_RATE, tempsc) if npas else (1, tempsc)
    O = Oracle(oracle_config(p, eos=eos))
    O.set_cooling(ck, tab, tempsc, psc, tsc)
    O.set_u(u0)
    O.boundaryI()
    O.calcprim_u()
    with _capi.Subdomain(p) as dev:
        dev.set_eos(*eos)
        dev.set_cooling(ck, tab, tempsc, psc, tsc)
        dev.upload_u(u0)
        for _ in range(2):
            dt = 0.1 * O.cfl_dtp()
            O.tstep(dt)
            dev.tstep(dt)
            folded = dev.cfl_dtp()
            assert folded == dev.cfl_dtp()        # the second call reduces in a pass of its own
            if _ == 0:
                ud, uo = dev.download_u(), O.get_u()
    O.close()
    same = [0, 1, 2, 3, 5, 6, 7] + ([4] if kind == "cold-table" else [])
    for q in same:
        np.testing.assert_array_equal(ud[q], uo[q], err_msg=f"field {q}")
    for q in range(4, 8 + npas):
        np.testing.assert_allclose(ud[q], uo[q], rtol=1e-10, atol=0, err_msg=f"field {q}")
