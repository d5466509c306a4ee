"""Host-only answers of the kernel library's C ABI (include/msnh_hip.h): what a caller decides by before it lays out memory."""
import ctypes
import itertools

import pytest

from msnhnet_amd import hipabi as abi


def _first_layer(dtype, in_c, out_c, k, **kw):
    f = dict(batch=2, h=40, w=36, stride=1, pad=0, groups=1, dil=1, out_ld=(out_c + 7) // 8 * 8, residual=0, out_dtype=dtype)
    f.update(kw)
    ext = f["dil"] * (k - 1) + 1
    oh, ow = (f["h"] + 2 * f["pad"] - ext) // f["stride"] + 1, (f["w"] + 2 * f["pad"] - ext) // f["stride"] + 1
    return abi.ConvDesc(dtype, f["out_dtype"], f["batch"], f["h"], f["w"], in_c, in_c, out_c, oh, ow, f["out_ld"], k, f["stride"], f["pad"], f["dil"], f["groups"], abi.ACT["none"], 0.1,
                        f["residual"], out_c, abi.ACT["none"], 0.1, 1.0, 1.0, abi.ALGO["auto"], 0, 0, 0)


@pytest.mark.parametrize("dtype", [abi.F32, abi.F16])
def test_auto_reads_nchw_for_multiples_of_32_filters_only(dtype):
    """AUTO's choice says what the caller's input has to be: STEM reads NCHW float32, everything else NHWC in the descriptor's type.  The filter counts
    that STEM has learned since must be asked for"""
    L = abi.lib()
    for in_c, out_c, k, stride in itertools.product((1, 2, 3, 4), (8, 16, 24, 32, 48, 64, 96), (1, 3, 5, 7), (1, 2)):
        d = _first_layer(dtype, in_c, out_c, k, stride=stride)
        auto, stem = L.msnh_hip_conv2d_select_algo(ctypes.byref(d)), L.msnh_hip_conv2d_stem_supported(ctypes.byref(d))
        assert (auto == abi.ALGO["stem"]) == (out_c % 32 == 0), (in_c, out_c, k)
        assert stem == (1 if out_c % 32 == 0 or (out_c == 16 and k >= 3 and k * k * in_c <= 160) else 0), (in_c, out_c, k)
        d.algo = abi.ALGO["stem"]
        assert L.msnh_hip_conv2d_select_algo(ctypes.byref(d)) == abi.ALGO["stem"]


def test_stem_refuses_what_it_cannot_run():
    L = abi.lib()
    ok = lambda d: L.msnh_hip_conv2d_stem_supported(ctypes.byref(d))
    assert ok(_first_layer(abi.F16, 3, 16, 3)) == 1 and ok(_first_layer(abi.F32, 3, 32, 7)) == 1
    for d in (_first_layer(abi.F16, 8, 32, 3), _first_layer(abi.F16, 3, 16, 3, out_dtype=abi.F32), _first_layer(abi.F32, 3, 32, 3, residual=1), _first_layer(abi.F32, 3, 32, 3, dil=2),
              _first_layer(abi.F16, 3, 16, 3, out_ld=18), _first_layer(abi.F16, 3, 16, 9)):
        assert ok(d) == 0
    assert L.msnh_hip_conv2d_stem_supported(None) == 0


@pytest.mark.parametrize("dtype", [abi.F32, abi.F16])
def test_focus_opening_is_asked_for(dtype):
    L = abi.lib()
    for in_c, out_c in itertools.product((1, 2, 3, 4), (8, 16, 32, 48, 64, 96, 128)):
        d = _first_layer(dtype, in_c, out_c, 6, stride=2, pad=2)
        auto = L.msnh_hip_conv2d_select_algo(ctypes.byref(d))
        assert auto != abi.ALGO["stem_focus"] and (auto == abi.ALGO["stem"]) == (out_c % 32 == 0)
        d.algo = abi.ALGO["stem_focus"]
        takes = in_c <= 3 and (out_c in (16, 32, 64, 128) or (out_c == 96 and dtype == abi.F32))
        assert L.msnh_hip_conv2d_stem_supported(ctypes.byref(d)) == takes, (in_c, out_c)
        assert (L.msnh_hip_conv2d_packed_weight_elems(ctypes.byref(d), d.algo) > 0) == takes
        d.ksize, d.pad = 5, 2
        assert L.msnh_hip_conv2d_stem_supported(ctypes.byref(d)) == 0


@pytest.mark.parametrize("dtype", [abi.F32, abi.F16])
def test_tiles_to_slice_take_slices(dtype):
    """the configurations that the library names for sliced launches exist and take slices of a small, deep layer in both types; the upsampling epilogue
    goes with unsliced launches only"""
    L = abi.lib()
    n = L.msnh_hip_conv2d_sliced_tiles(None, 0)
    tiles = (ctypes.c_int * (n + 1))(*([-7] * (n + 1)))
    assert L.msnh_hip_conv2d_sliced_tiles(tiles, n) == n and tiles[n] == -7
    one = (ctypes.c_int * 2)(-7, -7)
    assert L.msnh_hip_conv2d_sliced_tiles(one, 1) == n and (one[0], one[1]) == (tiles[0], -7)
    assert len(set(tiles[:n])) == n and all(1 <= t <= L.msnh_hip_conv2d_tile_count() for t in tiles[:n])
    for t in tiles[:n]:
        d = abi.ConvDesc(dtype, dtype, 1, 13, 13, 512, 512, 256, 13, 13, 256, 3, 1, 1, 1, 1, abi.ACT["leaky"], 0.1, 0, 256, abi.ACT["none"], 0.1, 1.0, 1.0, abi.ALGO["igemm_fusedk"], t + 256 * 4, 0, 0)
        assert L.msnh_hip_conv2d_tile_supported(ctypes.byref(d), d.tile) == 1, t
        assert L.msnh_hip_conv2d_workspace_bytes(ctypes.byref(d), d.algo) > 65536
        d.out_upsample = 2
        assert L.msnh_hip_conv2d_tile_supported(ctypes.byref(d), d.tile) == 0
