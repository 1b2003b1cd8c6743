"""What the entries of libhydra_mix.so refuse on the host, before anything is launched."""
import ctypes

import pytest


@pytest.mark.parametrize("n_tokens", [1, 2, 5, 100])
@pytest.mark.parametrize("mode", [3, -1])
def test_state_scan_refuses_an_unknown_recurrence(mode, n_tokens):
    from hydrainfer_amd import _lib
    buf = ctypes.create_string_buffer(1 << 16)
    at = ctypes.addressof(buf)
    a = _lib.hxm_state_scan_args(out=at, q=at, k=at, v=at, q_stride=64, k_stride=64, v_stride=64, decay=at, state=at, slot_stride=4096, slots=at, q_cu=at,
                                 positions=at, n_tokens=n_tokens, n_seq=1, heads=1, qk_heads=1, dim=64, vdim=64, mode=mode)
    HX_ERR_UNSUPPORTED = -5
    assert _lib.mix_lib().hxm_state_scan(ctypes.byref(a), None) == HX_ERR_UNSUPPORTED


@pytest.mark.parametrize("rows, experts, n, k, tile", [
    (1, 8, 2816, 2048, 32), (256, 8, 2816, 2048, 32), (768, 8, 2816, 2048, 128), (7976, 16, 4096, 2752, 256), (15956, 16, 5504, 4096, 256),
    # the measured best by more than a tenth (us in tiles of 64 / 128 / 256): 61 76 35, 86 104 54, 74 86 51, 48 60 33; 36 28 48; 35 28 48, 36 28 48
    (64 * 140, 64, 1024, 704, 256), (64 * 140, 64, 1024, 1408, 256), (32 * 140, 32, 2048, 1408, 256), (32 * 140, 32, 2048, 704, 256), (8 * 110, 8, 2816, 2048, 128),
    (16 * 80, 16, 1408, 2048, 128), (16 * 110, 16, 1408, 2048, 128),
    # 22 26 47, 43 55 57, 16 20 32
    (8 * 50, 8, 2816, 2048, 64), (16 * 50, 16, 2816, 2048, 64), (8 * 57, 8, 2048, 1408, 64)])
def test_tiles_of_the_grouped_product(rows, experts, n, k, tile):
    from hydrainfer_amd import _lib
    assert _lib.mix_lib().hxm_grouped_linear_tile_rows(rows, experts, n, k) == tile
