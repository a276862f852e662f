"""The launch shape a batch takes from its boxes' total work: boxes whose
corrector tiles (one a plane at 4 x 4 x nz) sum to either side of the lines
between the stage kernels, and a box admitted later that moves the batch over
one, equal the single-box path, bit for bit."""
import sys

import numpy as np
import pytest

from guacho_amd import _capi
from tests._pairs import random_state
from tests.test_gpu_batch import single

pytestmark = pytest.mark.gpu

FP64, MIXED = _capi.GM_PRECISION_FP64, _capi.GM_PRECISION_MIXED


def _box(nz, npas, prec):
    p = _capi.make_params(4, 4, nz, 0.25, 0.25, 0.25, bc=(1, 1, 2, 2, 3, 3), npas=npas, precision=prec)
    return p, random_state(np.random.default_rng(nz + npas), 4, 4, nz, npas=npas)


@pytest.mark.parametrize("prec,npas,first,later", [
    (FP64, 0, (300, 212), 0), (FP64, 0, (300, 213), 0), (FP64, 0, (300, 100), 300), (FP64, 0, (32000, 5), 800),
    (FP64, 1, (200, 56), 0), (FP64, 1, (200, 57), 0), (FP64, 2, (200, 3), 100),
    (MIXED, 0, (300, 213), 30), (MIXED, 1, (300, 84), 0), (MIXED, 1, (300, 85), 0), (MIXED, 2, (300, 3), 100)])
def test_batch_shape(prec, npas, first, later):
    print(f"case: batch shape, precision {prec}, {npas} passive scalars, nz {first}, then {later}", flush=True)
    sys.stdout.flush()
    bx = [_box(nz, npas, prec) for nz in first]
    with _capi.Batch(precision=prec, max_boxes=4, steps_per_launch=2) as B:
        ids = [B.add(p, u, max_steps=4) for p, u in bx]
        B.advance(1)
        B.sync()
        if later:
            bx.append(_box(later, npas, prec))
            ids.append(B.add(*bx[-1], max_steps=4))
        B.advance(2)
        B.sync()
        got = [B.download_u(i) for i in ids]
    for (p, u), g in zip(bx, got):
        np.testing.assert_array_equal(g, single(p, u, nsteps=4)[0])
