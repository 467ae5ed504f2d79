"""A red-black scene on a device with room for one ping-pong field but not for
three runs its diffusions one after the other."""
import ctypes

import numpy as np
import pytest

from equilibrium_amd import _abi
from helpers import assert_bit_equal

pytestmark = pytest.mark.gpu


def _frames(s, fields):
    for i, f in enumerate(fields):
        s.upload(i, f)
    s.step(2)
    s.sync()
    return [s.download(i) for i in range(6)]


def test_redblack_scene_where_three_pingpong_fields_do_not_fit():
    print("[case] red-black scene on a nearly full device", flush=True)
    hip = ctypes.CDLL("libamdhip64.so")
    p = _abi.default_params()
    p.size, p.gs_mode, p.gs_iters, p.pressure_iters = 3072, _abi.GS_REDBLACK, 7, 4
    p.delta_t, p.viscosity, p.diffusion = 0.1, 1e-6, 1e-6
    rng = np.random.default_rng(4)
    fields = [rng.standard_normal(p.size ** 2).astype(np.float32) for _ in range(6)]
    s = _abi.Scene(p)
    want = _frames(s, fields)
    s.close()
    # six fields of 36 MB and the rule bytes, one ping-pong field, the mask: 271 MB; three: 343
    mb, hogs = 1 << 20, []

    def fill(size):
        while True:
            q = ctypes.c_void_p()
            if hip.hipMalloc(ctypes.byref(q), ctypes.c_size_t(size * mb)) != 0:
                return hip.hipGetLastError()
            hogs.append((q, size))

    try:
        fill(8192)
        assert hip.hipFree(hogs.pop()[0]) == 0
        fill(64)
        gap = [hogs.pop() for _ in range(5)]
        fill(16)
        for q, _ in gap:  # 320 MB and less than a piece of 16
            assert hip.hipFree(q) == 0
        s = _abi.Scene(p)
        got = _frames(s, fields)
        q = ctypes.c_void_p()
        assert hip.hipMalloc(ctypes.byref(q), ctypes.c_size_t(72 * mb)) != 0  # (three would have fitted)
        hip.hipGetLastError()
        s.close()
    finally:
        for q, _ in hogs:
            assert hip.hipFree(q) == 0
    for k, (g, w) in enumerate(zip(got, want)):
        assert_bit_equal(g, w, f"field {k}")
