"""The slice-batched forward projection against the oracle: slice groups,
blocks of 64 and 128 rays, row bands, angles in any order and section, and rays
whose windows do not fit LDS or whose strips are many columns wide."""

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
GOLDEN = np.arange(311) * 2.399963229728653

# (geometry, image, slices, angles, detectors, dtype, order, further settings);
# at least 3e7 pixel-angles, a fan's detectors more than 512
STACKS = [
    ("radon", (129, 63), 3, 1300, 145, F32, "C", {}),      # an entry three quarters full, 3 ray blocks
    ("radon", (64, 64), 9, 900, 65, F32, "F", {}),         # one ray over, last slice alone
    ("radon", (200, 90), 5, 367, 513, F64, "F", {}),       # blocks of 128 rays, two entries
    ("radon", (96, 96), 2, 1700, 140, F64, "C", {}),
    ("fan", (160, 130), 8, 200, 641, F32, "F", {}),        # two entries, one ray over
    ("fan", (130, 160), 3, 500, 600, F32, "C", {}),
    ("fan", (110, 110), 11, 240, 520, F64, "C", {}),
    ("radon", (150, 150), 5, GOLDEN, 213, F32, "F", {}),   # angles in no order
    ("fan", (150, 150), 5, GOLDEN, 530, F64, "F", {}),
    ("radon", (150, 150), 5, [(150, 0.1, 0.6), (151, 2.0, 2.2)], 213, F64, "F", {}),
    ("radon", (128, 128), 8, 240, 23, F32, "F", {}),       # strips many columns wide
    ("radon", (1600, 90), 3, 140, 64, F32, "F", {}),       # windows wider than LDS
    ("fan", (300, 40), 8, 320, 540, F32, "F", dict(detector_width=9000.0)),  # a fan of 150 degrees
    ("fan", (40, 40), 8, 2400, 520, F64, "F", dict(detector_width=1200.0)),
    ("fan", (128, 128), 8, 260, 600, F32, "C", dict(midpoint_shift=(9.0, -14.0), detector_shift=11.0,
                                                    reverse_detector=True)),
    ("radon", (128, 128), 8, 260, 200, F64, "C", dict(midpoint_shift=(9.0, -14.0), detector_shift=11.0)),
]


def _settings(geometry, shape, angles, nd, more):
    n = float(max(shape))
    if geometry == "fan":
        kw = dict(R=2.0 * n, RE=n, image_width=n, detector_width=2.0 * n)
        return gratopy.ProjectionSettings("cuda:0", gratopy.FANBEAM, shape, angles, nd, **{**kw, **more})
    kw = dict(image_width=n, detector_width=2.0 ** 0.5 * n)
    return gratopy.ProjectionSettings("cuda:0", gratopy.RADON, shape, angles, nd, **{**kw, **more})


@pytest.mark.parametrize("geometry,shape,nz,angles,nd,dtype,order,more", STACKS)
def test_stack_forward_against_the_oracle(geometry, shape, nz, angles, nd, dtype, order, more):
    print(f"stack forward {geometry} {shape} x {nz}, {nd} det, {dtype}, {order}, {more}", flush=True)
    before = autotune.current_variant()
    try:
        autotune.set_variant(automatic=1)
        ps = _settings(geometry, shape, angles, nd, more)
        assert shape[0] * shape[1] * nz * ps.n_angles >= 3e7
        rng = np.random.default_rng(37)
        img = np.require(rng.random(shape + (nz,)).astype(dtype), requirements=order)
        sino = gratopy.forwardprojection(dev.to_device(img, "cuda:0", order=order), ps)
        torch.cuda.synchronize()
        got = dev.to_host(sino)
        for z in sorted({0, 1, nz // 2, nz - 1}):
            ref = _oracle(ps, img[:, :, z].astype(F64), F64, False)
            bar = TOL[dtype]
            if dtype == F32:
                bar = max(bar, 1.2 * rel_err(_oracle(ps, img[:, :, z], F32, False), ref))
            assert rel_err(got[:, :, z], ref) <= bar, z
    finally:
        autotune.set_variant(**before)


@pytest.mark.parametrize("geometry", ["radon", "fan"])
@pytest.mark.parametrize("value", [np.inf, np.nan, np.finfo(F32).max])
def test_values_off_a_rays_strip_do_not_reach_it(geometry, value):
    """A pixel that is not finite reaches exactly the bins whose strips hold it."""
    print(f"stack forward {geometry}, one pixel {value}", flush=True)
    before = autotune.current_variant()
    try:
        autotune.set_variant(automatic=1)
        ps = _settings(geometry, (128, 120), 250, 540, {})
        img = np.zeros((128, 120, 8), dtype=F32, order="F")
        img[40, 71, 5] = 1
        touched = dev.to_host(gratopy.forwardprojection(dev.to_device(img, "cuda:0"), ps)) != 0
        img[40, 71, 5] = value
        got = dev.to_host(gratopy.forwardprojection(dev.to_device(img, "cuda:0"), ps))
        assert np.all(got[~touched] == 0)
        assert np.all(got[touched] != 0)
    finally:
        autotune.set_variant(**before)
