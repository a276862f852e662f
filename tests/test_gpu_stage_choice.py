"""The choice of a step's stage kernels by corrector tiles (32 x 16 x 1, so nz
of them on a 4 x 4 x nz grid) and passive scalars, on both sides of each of its
lines: one step through the default kernels equals the restatement's, bit for
bit, and the mixed form's equals its own two-kernel stages, bit for bit."""
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from tests._pairs import random_state, run_pair

pytestmark = pytest.mark.gpu


def _box(nz, npas, precision):
    u0 = random_state(np.random.default_rng(nz + npas), 4, 4, nz, npas=npas)
    p = _capi.make_params(4, 4, nz, 0.25, 0.25, 0.25, bc=(3, 3, 1, 1, 3, 3), npas=npas, precision=precision)
    return u0, p


@pytest.mark.parametrize("nz,npas", [(512, 0), (513, 0), (32767, 0), (32768, 0), (256, 1), (257, 1), (256, 2), (257, 2)])
def test_stage_kernels_fp64(nz, npas):
    print(f"case: FP64 stage kernels, 4x4x{nz}, {npas} passive scalars, 1 step", flush=True)
    sys.stdout.flush()
    u0, p = _box(nz, npas, _capi.GM_PRECISION_FP64)
    ud, uo, _ = run_pair(p, u0, 1)
    np.testing.assert_array_equal(ud, uo)


@pytest.mark.parametrize("nz,npas", [(513, 0), (384, 1), (385, 1), (384, 2), (385, 2)])
def test_stage_kernels_mixed(nz, npas, monkeypatch):
    print(f"case: mixed stage kernels, 4x4x{nz}, {npas} passive scalars, 2 steps", flush=True)
    sys.stdout.flush()
    u0, p = _box(nz, npas, _capi.GM_PRECISION_MIXED)

    def run():
        with _capi.Subdomain(p) as dev:
            dev.upload_u(u0)
            for _ in range(2):
                dev.tstep(0.2 * dev.cfl_dtp())
            return dev.download_u()
    got = run()
    monkeypatch.setenv("GUACHO_AMD_SLAB_STAGES", "")
    np.testing.assert_array_equal(got, run())
    assert np.isfinite(got).all() and np.abs(got - u0)[:, 2:-2, 2:-2, 2:-2].max() > 1e-3
