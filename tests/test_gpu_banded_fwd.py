"""The automatic banded forward against the oracle: both group widths and every
band count, thin images whose bands hold a row or none, single bins and part
groups, two slices, wide fans whose groups leave their frame; and calls given a
workspace that holds only their general launch shape."""

from __future__ import annotations

import ctypes

import numpy as np
import pytest
import torch

import gratopy_amd as gratopy
from gratopy_amd import _device as dev
from gratopy_amd import _hip, autotune
from tests.helpers import rel_err
from tests.test_gpu_projection import TOL, _oracle
from tests.test_gpu_stack_fwd import _settings

pytestmark = pytest.mark.gpu

F32, F64 = np.dtype("float32"), np.dtype("float64")

# (geometry, image, slices, angles, detectors, dtype, order, further settings);
# single slices of at least 8e6 pixel-angles
CALLS = [
    ("radon", (199, 210), 1, 200, 300, F32, "F", {}),    # 16 bands
    ("radon", (201, 200), 1, 201, 17, F32, "C", {}),     # 32; a bin over a pair of groups
    ("fan", (479, 480), 1, 60, 500, F64, "F", {}),       # 32 bands, 8 bins
    ("fan", (481, 480), 1, 300, 512, F32, "C", {}),      # 48 bands, 16 bins
    ("radon", (480, 500), 1, 900, 513, F32, "F", {}),
    ("radon", (20, 2000), 1, 250, 600, F64, "F", {}),    # bands of one row or two
    ("fan", (3000, 9), 1, 320, 700, F32, "F", {}),       # empty bands
    ("fan", (300, 290), 2, 400, 1, F32, "C", {}),        # a single bin
    ("radon", (256, 256), 2, 200, 391, F32, "F", {}),
    ("fan", (230, 230), 1, 170, 345, F32, "F", dict(detector_width=1840.0)),  # half angle 63 degrees
    ("fan", (300, 300), 1, 100, 100, F64, "F", dict(detector_width=9000.0)),  # 82 degrees
]


@pytest.mark.parametrize("geometry,shape,nz,angles,nd,dtype,order,more", CALLS)
def test_banded_forward_against_the_oracle(geometry, shape, nz, angles, nd, dtype, order, more):
    print(f"banded forward {geometry} {shape} x {nz}, {angles} angles, {nd} det, {dtype}, {order}, {more}", flush=True)
    before = autotune.current_variant()
    try:
        autotune.set_variant(automatic=1)
        ps = _settings(geometry, shape, angles, nd, more)
        z = (nz,) if nz > 1 else ()
        img = np.require(np.random.default_rng(43).random(shape + z).astype(dtype), requirements=order)
        d_img = dev.to_device(img, "cuda:0", order=order)
        got = dev.to_host(gratopy.forwardprojection(d_img, ps)).reshape(nd, angles, nz)
        # the entry point without allocations takes the route its array holds
        small = dev.zeros((nd, angles) + z, dtype, order="F", device="cuda:0")
        tables = [ps.ofs_buf[dtype], ps.sdpd_buf[dtype] if ps.is_fan else None, ps.geometry_information[dtype]]
        _hip.call("gt_projection_noalloc", torch.cuda.current_stream().cuda_stream, int(ps.is_fan), 0,
                  _hip.dtype_code(dtype), small.data_ptr(), d_img.data_ptr(),
                  tables[0].data_ptr(), tables[1].data_ptr() if ps.is_fan else None, tables[2].data_ptr(),
                  *shape, nd, angles, nz, 0, dev.order_code(order))
        torch.cuda.synchronize()
        for result in (got, dev.to_host(small).reshape(nd, angles, nz)):
            for k in range(nz):
                x = img.reshape(shape + (nz,))[:, :, k]
                ref = _oracle(ps, x.astype(F64), F64, False)
                bar = TOL[dtype]
                if dtype == F32:
                    bar = max(bar, 1.2 * rel_err(_oracle(ps, x, F32, False), ref))
                assert rel_err(result[:, :, k], ref) <= bar, k
    finally:
        autotune.set_variant(**before)


@pytest.mark.parametrize("adjoint", [0, 1])
@pytest.mark.parametrize("geometry,shape,nz,angles,nd", [
    ("fan", (300, 310), 1, 200, 400), ("radon", (500, 490), 1, 300, 700),
    ("radon", (64, 64), 9, 900, 65), ("fan", (160, 130), 8, 200, 641)])
def test_a_workspace_of_the_general_shape_suffices(geometry, shape, nz, angles, nd, adjoint):
    print(f"general workspace {geometry} {shape} x {nz}, adjoint {adjoint}", flush=True)
    before = autotune.current_variant()
    lib = _hip.load_library()
    try:
        ps = _settings(geometry, shape, angles, nd, {})
        ps.ensure_dtype(F32)
        sizes = (*shape, nd, angles, nz)
        autotune.set_variant(automatic=1)
        full = lib.gt_projection_workspace_bytes(int(ps.is_fan), adjoint, 0, *sizes, 0)
        knobs = (ctypes.c_int * 4)()
        assert lib.gt_projection_shape(int(ps.is_fan), adjoint, *sizes, knobs) == _hip.GT_OK
        names = (("back_rows", "back_bands", "back_stage", "back_tile") if adjoint else
                 ("fwd_group", "fwd_bands", "fwd_chunk", "fwd_compact"))
        autotune.set_variant(**dict(zip(names, list(knobs))))
        general = lib.gt_projection_workspace_bytes(int(ps.is_fan), adjoint, 0, *sizes, 0)
        autotune.set_variant(automatic=1)
        nin, nout = (ps.sinogram_shape, shape) if adjoint else (shape, ps.sinogram_shape)
        x = np.asfortranarray(np.random.default_rng(47).random(tuple(nin) + (nz,)).astype(F32))
        arg = dev.to_device(x, "cuda:0")
        out = dev.zeros(tuple(nout) + (nz,), F32, device="cuda:0")
        tables = [ps.ofs_buf[F32].data_ptr()] + ([ps.sdpd_buf[F32].data_ptr()] if ps.is_fan else [])
        tables.append(ps.geometry_information[F32].data_ptr())
        name = f"gt_{geometry}_{'back' if adjoint else 'fwd'}"
        ref = [_oracle(ps, x[:, :, k].astype(F64), F64, bool(adjoint)) for k in (0, nz - 1)]
        for size in {general, max(general, full)}:
            ws = torch.empty(size, dtype=torch.uint8, device="cuda:0")
            args = (torch.cuda.current_stream().cuda_stream, 0, out.data_ptr(), arg.data_ptr(), *tables, *sizes, 0, 0)
            _hip.call(name, *args, ws.data_ptr(), size)
            torch.cuda.synchronize()
            got = dev.to_host(out)
            for k, r in zip((0, nz - 1), ref):
                bar = max(TOL[F32], 1.2 * rel_err(_oracle(ps, x[:, :, k], F32, bool(adjoint)), r))
                assert rel_err(got[:, :, k], r) <= bar, (size, k)
        assert getattr(lib, name)(*args, ws.data_ptr(), general - 1) == _hip.GT_ENOSPC
    finally:
        autotune.set_variant(**before)
