"""Readback through the pinned ring: arrays of less than one chunk (2^21 source
bytes), one more and one less than whole chunks, and more than the ring holds,
in every width the device keeps, into fresh, offset and pinned host memory.

A field loaded from the host comes back as loaded, rounded to what the form
holds (float for E, H, Q; 2^-40 fixed point for the FP32 form's current)."""
import ctypes as C
import importlib

import numpy as np
import pytest

pytestmark = pytest.mark.gpu

pic = importlib.import_module("0buf_amd")

#  ghosted nodes: 216; 2^18 and 2^19 exactly (one chunk of 8 and of 4 byte
#  elements); one layer more; 2.2 million (over 8 chunks of doubles)
BOXES = [(4, 4, 4), (62, 62, 62), (62, 62, 126), (63, 62, 126), (128, 128, 128)]


@pytest.mark.parametrize("n", BOXES)
@pytest.mark.parametrize("precision", [pic.FP64, pic.FP32])
def test_fields_come_back_as_loaded(n, precision):
    g = pic.Pic(pic.make_params(n, tuple(0.1 * k for k in n), 0.05, precision=precision))
    rng = np.random.default_rng(n[2] + precision)
    for which in (0, 4, 6, 11):
        a = rng.normal(0.0, 1.0, g.G)
        g.load_field(which, a)
        want = a
        if precision == pic.FP32:
            want = np.rint(a * 2.0**40) * 2.0**-40 if 6 <= which <= 8 else a.astype(np.float32)
        assert np.array_equal(g.get_field(which), want), which
    # into memory at an odd offset, and into pinned memory
    import torch
    for buf in (np.full(g.G + 3, -1.0), torch.full((g.G + 3,), -1.0, dtype=torch.float64,
                                                   pin_memory=True).numpy()):
        out = buf[1:g.G + 1]
        assert g.lib.pic_get_field(g._ctx, 11, out.ctypes.data_as(C.POINTER(C.c_double))) == 0
        assert np.array_equal(out, want)
        assert buf[0] == -1.0 and buf[g.G + 1] == -1.0 and buf[g.G + 2] == -1.0
    g.close()


@pytest.mark.parametrize("precision", [pic.FP64, pic.FP32])
def test_particles_and_counts_of_many_chunks(precision):
    n = (96, 96, 64)                     # 589,824 cells, over one chunk of counts
    g = pic.Pic(pic.make_params(n, tuple(0.1 * k for k in n), 0.05, precision=precision))
    rng = np.random.default_rng(3)
    P = 300_001
    x = [rng.uniform(0.0, 0.1 * k * (1 - 1e-9), P) for k in n]
    cell = np.ravel_multi_index([np.floor(v / 0.1).astype(int) for v in x], n)
    g.load_particles(1, *x, *(np.zeros(P) for _ in range(3)), -1.0, -1.0)
    counts = g.cell_counts()
    assert counts.sum() == P
    assert np.abs(counts - np.bincount(cell, minlength=counts.size)).sum() <= 4   # at faces
    p = g.particles()
    assert np.array_equal(np.bincount(p["cell"], minlength=counts.size), counts)
    tol = 1e-14 if precision == pic.FP64 else 0.1 * 2.0**-23
    assert np.abs(np.sort(p["x"]) - np.sort(x[0])).max() <= tol
    assert np.array_equal(g.cell_moments(1, "density"), -1.0 * counts)
    g.close()
