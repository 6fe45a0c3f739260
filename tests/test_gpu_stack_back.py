"""The slice-batched backprojection against the oracle, at the edges of its
tiles (32 x 16 and 32 x 32 pixels), window tables (128 angles), slice groups
(4 or 2 slices per entry, one or two entries per lane) and staged windows."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gratopy_amd as gratopy
from gratopy_amd import _device as dev
from gratopy_amd import autotune
from tests.helpers import rel_err
from tests.test_gpu_projection import TOL, _oracle

pytestmark = pytest.mark.gpu

F32, F64 = np.dtype("float32"), np.dtype("float64")

# (geometry, image, slices, angles, detectors, dtype, order); at least 2e7 pixel-angles
STACKS = [
    ("fan", (33, 47), 9, 1500, 70, F32, "C"),      # one entry per lane, a last slice alone
    ("radon", (32, 16), 8, 5000, 50, F32, "F"),    # exactly one tile, two entries
    ("fan", (65, 31), 16, 700, 97, F32, "F"),      # one column and one row over
    ("radon", (100, 129), 3, 521, 182, F32, "C"),  # an entry three quarters full
    ("fan", (64, 64), 2, 2500, 90, F64, "F"),      # float64: two slices per entry
    ("radon", (31, 90), 5, 1440, 100, F64, "C"),
    ("fan", (40, 40), 4, 3200, 2400, F32, "F"),    # every window too wide to stage
    ("radon", (64, 64), 8, 650, 704, F32, "F"),    # some windows too wide
    ("fan", (64, 64), 8, 650, 704, F64, "C"),
    ("radon", (256, 256), 192, 5, 300, F32, "F"),  # four pixels per lane
    ("fan", (256, 256), 97, 5, 300, F64, "F"),
]


def _settings(geometry, shape, na, nd):
    n = float(max(shape))
    if geometry == "fan":
        return gratopy.ProjectionSettings("cuda:0", gratopy.FANBEAM, shape, na, nd, R=2.0 * n, RE=n,
                                          image_width=n, detector_width=2.0 * n)
    return gratopy.ProjectionSettings("cuda:0", gratopy.RADON, shape, na, nd)


@pytest.mark.parametrize("geometry,shape,nz,na,nd,dtype,order", STACKS)
def test_stack_backprojection_against_the_oracle(geometry, shape, nz, na, nd, dtype, order):
    print(f"stack back {geometry} {shape} x {nz}, {na} angles, {nd} det, {dtype}, {order}", flush=True)
    before = autotune.current_variant()
    try:
        autotune.set_variant(automatic=1)
        ps = _settings(geometry, shape, na, nd)
        rng = np.random.default_rng(31)
        sino = np.require(rng.random((nd, na, nz)).astype(dtype), requirements=order)
        back = gratopy.backprojection(dev.to_device(sino, "cuda:0", order=order), ps)
        torch.cuda.synchronize()
        got = dev.to_host(back)
        for z in sorted({0, 1, nz // 2, nz - 1}):
            ref = _oracle(ps, sino[:, :, z].astype(F64), F64, True)
            bar = TOL[dtype]
            if dtype == F32:
                bar = max(bar, 1.2 * rel_err(_oracle(ps, sino[:, :, z], F32, True), ref))
            assert rel_err(got[:, :, z], ref) <= bar, z
    finally:
        autotune.set_variant(**before)
