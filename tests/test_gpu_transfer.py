"""Uploads and downloads through the pinned staging ring, bit for bit: arrays
below and above the size from which it is taken, an exact number of its 8 MiB
chunks and a ragged last one, in FP64; primitives, temperature and div B of
the larger one; two threads with a context each, of which one finds the ring
in use; and batch boxes whose device block served another box before (same
size, slightly smaller, and larger than any spare one)."""
import threading

import numpy as np
import pytest

from guacho_amd import _capi
from tests._pairs import random_state

pytestmark = pytest.mark.gpu


def params(n):
    return _capi.make_params(*n, 1.0 / n[0], 1.0 / n[1], 1.0 / n[2], bc=(1,) * 6)


def inner(u):
    return u[:, 2:-2, 2:-2, 2:-2]


# (nx+4)(ny+4)(nz+4) * 64 bytes: 16 MiB less one plane, 16 MiB = 2 chunks, 24 MiB + 12 KiB
SIZES = [(60, 60, 59), (60, 60, 60), (60, 60, 92), (61, 60, 92)]


@pytest.mark.parametrize("n", SIZES, ids=lambda n: "x".join(map(str, n)))
def test_round_trip(n):
    print(f"case: upload and download {n}", flush=True)
    rng = np.random.default_rng(sum(n))
    with _capi.Subdomain(params(n)) as dev:
        for _ in range(2):
            u = random_state(rng, *n)
            dev.upload_u(u)
            np.testing.assert_array_equal(inner(dev.download_u()), inner(u))
        p, t = dev.download_primit(with_temp=True)
        np.testing.assert_array_equal(p[0], np.maximum(dev.download_u()[0], 1e-15))
        assert np.isfinite(t).all() and dev.divb().shape == n


def test_two_threads():
    print("case: two threads, a context each, 8 round trips at 60x60x92", flush=True)
    n, bad = SIZES[2], []

    def work(seed):
        rng = np.random.default_rng(seed)
        with _capi.Subdomain(params(n)) as dev:
            for _ in range(8):
                u = random_state(rng, *n)
                dev.upload_u(u)
                if not np.array_equal(inner(dev.download_u()), inner(u)):
                    bad.append(seed)
    threads = [threading.Thread(target=work, args=(s,)) for s in (1, 2)]
    for t in threads:
        t.start()
    for t in threads:
        t.join()
    assert not bad


def test_boxes_on_reused_blocks():
    print("case: batch boxes on blocks of released boxes", flush=True)
    rng = np.random.default_rng(5)
    sizes = [(20, 20, 20), (20, 20, 20), (20, 20, 19), (24, 20, 20), (20, 20, 20)]
    boxes = [(params(n), random_state(rng, *n)) for n in sizes]
    alone = []
    for p, u in boxes:
        with _capi.Batch(precision=_capi.GM_PRECISION_FP64, max_boxes=1) as B:
            b = B.add(p, u, max_steps=3)
            B.advance(3)
            B.sync()
            alone.append(B.download_u(b))
    with _capi.Batch(precision=_capi.GM_PRECISION_FP64, max_boxes=2) as B:
        budget = B.free_bytes()
        for (p, u), want in zip(boxes, alone):
            b = B.add(p, u, max_steps=3)
            assert B.free_bytes() == budget - B.box_bytes(p)
            B.advance(3)
            B.sync()
            np.testing.assert_array_equal(B.download_u(b), want)
            B.remove(b)
            assert B.free_bytes() == budget
