"""One-launch projections of small calls against the oracle: fewer rows or
angles than waves, single bins, partial tiles and ray blocks, both sides of each
size rule, both memory orders on either side, stacks, windows wider than a wave's
LDS, rays that leave their block's frame, values that are not finite."""

from __future__ import annotations

import numpy as np
import pytest
import torch

import gratopy_amd as gratopy
from gratopy_amd import _device as dev
from gratopy_amd import autotune
from tests.helpers import rel_err
from tests.test_gpu_projection import TOL, _oracle
from tests.test_gpu_stack_fwd import _settings

pytestmark = pytest.mark.gpu

F32, F64 = np.dtype("float32"), np.dtype("float64")

# (geometry, image, slices, angles, detectors, dtype, further settings)
CALLS = [
    ("radon", (1, 1), 1, 1, 1, F32, {}),
    ("fan", (2, 1), 1, 3, 2, F64, {}),
    ("radon", (7, 5), 1, 17, 65, F32, {}),                # fewer rows than waves, one ray over
    ("fan", (9, 17), 2, 16, 64, F32, {}),                 # an angle a wave, tiles of one column or row
    ("radon", (64, 33), 1, 129, 91, F64, {}),
    ("fan", (100, 75), 1, 45, 130, F32, {}),
    ("fan", (75, 100), 3, 31, 130, F64, {}),
    ("radon", (101, 97), 1, [0.3, 2.9, 0.1, 1.6], 145, F32, {}),
    ("radon", (128, 128), 1, 121, 179, F32, {}),          # just below and above 2e6 pixel-angles
    ("radon", (128, 128), 1, 123, 179, F32, {}),
    ("fan", (128, 128), 1, 123, 179, F32, {}),
    ("fan", (64, 64), 6, 100, 90, F64, {}),
    ("radon", (230, 231), 1, 150, 280, F32, {}),          # just below and above 8e6
    ("fan", (231, 230), 1, 151, 300, F32, {}),
    ("fan", (256, 240), 1, 320, 360, F32, {}),            # just below 2e7
    ("radon", (300, 301), 1, 540, 420, F32, {}),          # just below 5e7
    ("radon", (64, 64), 1, 40, 9, F32, {}),               # strips many columns wide
    ("radon", (64, 64), 1, 40, 3000, F32, {}),            # many bins a pixel: windows wider than LDS
    ("fan", (150, 150), 1, 100, 1500, F64, {}),
    ("radon", (1200, 20), 1, 20, 30, F32, {}),
    ("fan", (40, 40), 1, 60, 60, F32, dict(detector_width=1200.0)),  # a fan of 150 degrees
    ("fan", (40, 40), 1, 60, 120, F64, dict(detector_width=1200.0)),
    ("fan", (40, 40), 1, 60, 60, F64, dict(RE=29.0)),     # tiles' corners beyond the source
    ("fan", (96, 64), 1, 60, 150, F32, dict(midpoint_shift=(9.0, -14.0), detector_shift=11.0,
                                            reverse_detector=True)),
]


def _auto(run):
    before = autotune.current_variant()
    try:
        autotune.set_variant(automatic=1)
        run()
    finally:
        autotune.set_variant(**before)


@pytest.mark.parametrize("orders", ["FF", "CC", "FC", "CF"])
@pytest.mark.parametrize("geometry,shape,nz,angles,nd,dtype,more", CALLS)
def test_small_calls_against_the_oracle(geometry, shape, nz, angles, nd, dtype, more, orders):
    print(f"small {geometry} {shape} x {nz}, {nd} det, {dtype}, {orders}, {more}", flush=True)

    def run():
        ps = _settings(geometry, shape, angles, nd, more)
        rng = np.random.default_rng(41)
        for adjoint in (False, True):
            nin, nout = (ps.sinogram_shape, ps.img_shape) if adjoint else (ps.img_shape, ps.sinogram_shape)
            z = (nz,) if nz > 1 else ()
            x = np.require(rng.random(tuple(nin) + z).astype(dtype), requirements=orders[0])
            out = dev.zeros(tuple(nout) + z, dtype, order=orders[1], device="cuda:0")
            arg = dev.to_device(x, "cuda:0", order=orders[0])
            if adjoint:
                gratopy.backprojection(arg, ps, img=out)
            else:
                gratopy.forwardprojection(arg, ps, sino=out)
            torch.cuda.synchronize()
            got = dev.to_host(out).reshape(tuple(nout) + (nz,))
            for k in {0, nz - 1}:
                xk = x.reshape(tuple(nin) + (nz,))[:, :, k]
                ref = _oracle(ps, xk.astype(F64), F64, adjoint)
                bar = TOL[dtype]
                if dtype == F32:
                    bar = max(bar, 1.2 * rel_err(_oracle(ps, xk, F32, adjoint), ref))
                assert rel_err(got[:, :, k], ref) <= bar, (adjoint, k)

    _auto(run)


@pytest.mark.parametrize("geometry", ["radon", "fan"])
@pytest.mark.parametrize("value", [np.inf, np.nan, np.finfo(F32).max])
def test_values_off_a_rays_strip_do_not_reach_it(geometry, value):
    """A pixel that is not finite reaches exactly the bins whose strips hold it."""
    print(f"small forward {geometry}, one pixel {value}", flush=True)

    def run():
        ps = _settings(geometry, (64, 50), 60, 100, {})
        img = np.zeros((64, 50), dtype=F32, order="F")
        img[20, 31] = 1
        touched = dev.to_host(gratopy.forwardprojection(dev.to_device(img, "cuda:0"), ps)) != 0
        img[20, 31] = value
        got = dev.to_host(gratopy.forwardprojection(dev.to_device(img, "cuda:0"), ps))
        assert np.all(got[~touched] == 0)
        assert np.all(got[touched] != 0)

    _auto(run)
