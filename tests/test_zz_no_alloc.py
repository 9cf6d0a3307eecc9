"""The allocation-free gendaymtx entry point (rg_sky_matrix_device_noalloc)
against the allocating one (rg_sky_matrix_device): the same kernels, so the
matrices are identical, on two calls in a row (the second smaller than the
first), through the C ABI; a plan larger than its fixed device array is
refused with an error."""

import ctypes as C
import json

import numpy as np
import pytest

from conftest import GOLDEN

pytestmark = pytest.mark.gpu


def _say(msg):
    print(msg, flush=True)


def test_noalloc_sky_matrix_matches_allocating_entry_point():
    import torch
    from pyradiance_amd import _lib, gen, scenes
    L = _lib.lib()
    fn = L.rg_sky_matrix_device_noalloc
    fn.argtypes = [C.c_void_p, C.c_void_p]
    fn.restype = C.c_int
    meta = json.loads((GOLDEN / "sky_cases.json").read_text())
    cases = [("annual tape, Reinhart MF:4, 8760 steps", scenes.annual_wea(3), ["-m", "4"]),
             ("wea1 tape, MF:1 with options", meta["tapes"]["wea1"], meta["cases"]["wea1_m2_opts"]["args"])]
    for name, tape, args in cases:
        _say(f"noalloc gendaymtx: {name}")
        mtx, sky, _, _ = gen.sky_matrix(tape, args)
        try:
            d_alloc = torch.full(mtx.shape, float("nan"), dtype=torch.float32, device="cuda")
            d_free = torch.full(mtx.shape, float("nan"), dtype=torch.float32, device="cuda")
            sky.matrix_device(d_alloc.data_ptr())
            assert fn(sky._h, C.c_void_p(d_free.data_ptr())) == 0, L.rg_sky_error(sky._h).decode()
            torch.cuda.synchronize()
            assert torch.equal(d_free, d_alloc)
            assert np.array_equal(d_free.cpu().numpy(), mtx)
        finally:
            sky.close()
    _say("noalloc gendaymtx: plan beyond the fixed array")
    mtx, sky, _, _ = gen.sky_matrix(scenes.annual_wea(3), ["-m", "4", "-A"])
    try:
        d = torch.empty(mtx.shape, dtype=torch.float32, device="cuda")
        assert fn(sky._h, C.c_void_p(d.data_ptr())) != 0
        assert "allocation-free" in L.rg_sky_error(sky._h).decode()
    finally:
        sky.close()


@pytest.mark.parametrize("args, most", [(["-m", "64"], 23), (["-m", "64", "-A", "-u"], 5)])
def test_noalloc_accepts_plans_up_to_the_last_step_its_array_holds(args, most):
    """Scratch of a plan: 76 bytes a patch (eight FP64 terms, three floats) and
    4 a patch and step, with -A 12 more a patch and step; at 144 * 64^2 + 2
    patches 96 MiB hold 23 steps, with -A 5 (steps and parts' padding take
    less than the rest).  One step, and with -A its one row of partial sums,
    is the other end."""
    import torch
    from pyradiance_amd import _lib
    from pyradiance_amd.gen import _parse_args

    def tape(n):
        return ("place X\nlatitude 37.0\nlongitude 122.0\ntime_zone 120\nsite_elevation 10\n"
                "weather_data_file_units 1\n" + "".join(f"6 {21 + i // 12} {6.5 + i % 12} {100 + i} {80 + i}\n" for i in range(n)))
    np_ = 144 * 64 ** 2 + 2
    per = 16 if "-A" in args else 4
    assert np_ * (76 + per * most) < 96 << 20 < np_ * (76 + per * (most + 1))
    for n in (1, 2, most):
        _say(f"noalloc gendaymtx: {' '.join(args)}, {n} steps")
        sky = _lib.Sky(tape(n), _parse_args(args)[0])
        try:
            assert sky.npatch == np_
            shape = (sky.npatch, sky.ncols, 3)
            d_alloc = torch.full(shape, float("nan"), dtype=torch.float32, device="cuda")
            d_free = torch.full(shape, float("nan"), dtype=torch.float32, device="cuda")
            sky.matrix_device(d_alloc.data_ptr())
            sky.matrix_device_noalloc(d_free.data_ptr())
            torch.cuda.synchronize()
            assert torch.equal(d_free, d_alloc) and bool(d_alloc.isfinite().all()) and bool((d_alloc > 0).any())
        finally:
            sky.close()
    sky = _lib.Sky(tape(most + 1), _parse_args(args)[0])
    try:
        with pytest.raises(Exception, match="allocation-free"):
            sky.matrix_device_noalloc(d_free.data_ptr())
    finally:
        sky.close()
