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
