"""The server's HBM budget: which requests it takes, and what a resident scene
really holds."""
import ctypes
import time

import numpy as np
import pytest

from equilibrium_amd import _abi, scenes
from helpers import assert_bit_equal, gpu_scene

pytestmark = pytest.mark.gpu

ENDED = (_abi.REQ_DONE, _abi.REQ_FAILED, _abi.REQ_CANCELLED)


def _accepted(S, mode):
    """The least budget that takes a request of this size: ten fields (red-black), or
    nine of whole strips of 64 rows and columns rounded up to 16, and what goes with them."""
    N, up = S - 2, lambda v, q: (v + q - 1) // q * q
    if mode == _abi.GS_REDBLACK:
        return 9 * up(S * S, 64) * 4 + up(S * (S + S % 2), 64) + 4 * S * S + 5 * S + 96 * N + 128 + 8192
    cells = up(N, 64) * up(N, 16)
    return 9 * up(cells + 4 * S, 64) * 4 + cells * 3 // 4 + S + 96 * N + 128 + 4096


def _free():
    hip = ctypes.CDLL("libamdhip64.so")
    f, t = ctypes.c_size_t(), ctypes.c_size_t()
    assert hip.hipMemGetInfo(ctypes.byref(f), ctypes.byref(t)) == 0
    return f.value


@pytest.mark.parametrize("S,mode", [(S, _abi.GS_WAVEFRONT) for S in (3, 34, 66, 130, 258, 322, 514)] +
                         [(S, _abi.GS_REDBLACK) for S in (66, 300, 1101)])
def test_least_budget_serves_its_scene(S, mode):
    """... with sources and obstacles, bit for bit as on its own, and one byte less refuses it."""
    print(f"[case] budget S={S} mode={mode}", flush=True)
    sc = scenes.stam_scene(S - 2, scenes.derive_seed(62, S), iters=20, frames=2, n_rects=0 if S < 40 else 2)
    least = _accepted(S, mode)
    srv = _abi.Server(least - 1)
    with pytest.raises(_abi.EqfError) as ei:
        srv.submit(sc, gs_mode=mode)
    assert ei.value.code == _abi.EQF_ENOMEM
    srv.close()
    srv = _abi.Server(least)
    ts = [srv.submit(sc, gs_mode=mode) for _ in range(3)]
    srv.wait_idle(60000)
    s = gpu_scene(sc, mode)
    s.step(2)
    s.sync()
    for t in ts:
        assert srv.poll(t).state == _abi.REQ_DONE
        assert_bit_equal(srv.result(t), s.download(_abi.DENSITY), f"S={S}")
    st = srv.stats()
    assert st["peak_bytes"] <= 1.11 * least  # a scene's own bytes are at most 1.102 times what the rule counts
    s.close()
    srv.close()


@pytest.mark.parametrize("mode", [_abi.GS_WAVEFRONT, _abi.GS_REDBLACK])
def test_resident_scene_holds_what_it_is_charged(mode):
    """A budget that one scene fills: the memory that goes while it is resident is
    what the server says (the pool takes it in larger pieces)."""
    N = 1000 if mode == _abi.GS_WAVEFRONT else 2900
    print(f"[case] charged bytes mode={mode}", flush=True)
    sc = scenes.stam_scene(N, scenes.derive_seed(63, N), iters=4, frames=10 ** 6, n_rects=1)
    warm = gpu_scene(sc, mode)  # what the process loads once
    warm.step(2)
    warm.sync()
    warm.close()
    budget = _accepted(N + 2, mode)
    srv = _abi.Server(budget)
    before = _free()
    t = srv.submit(sc, gs_mode=mode)
    for _ in range(20000):
        if srv.poll(t).frames_done > 1:
            break
        time.sleep(0.001)
    held = before - _free()
    st = srv.stats()
    srv.release(t)
    srv.wait_idle(60000)
    srv.close()
    print(f"[budget] {budget / 2**20:.1f} MiB, charged {st['peak_bytes'] / 2**20:.1f}, held {held / 2**20:.1f}", flush=True)
    assert held > 0.5 * budget
    assert st["peak_bytes"] <= 1.11 * budget
    assert held <= st["peak_bytes"] + (24 << 20)


def test_full_and_lean_scenes_share_a_tick():
    """Scenes with workspaces for three lin_solves and for one in one lane."""
    print("[case] full and lean scenes", flush=True)
    big = [scenes.stam_scene(240, scenes.derive_seed(64, i), iters=12, frames=12, n_rects=2) for i in range(2)]
    small = [scenes.stam_scene(N, scenes.derive_seed(65, N), iters=12, frames=6, n_rects=1) for N in (20, 33, 64)]
    srv = _abi.Server(_accepted(242, _abi.GS_WAVEFRONT) + (300 << 10))  # 240 has one, the small ones three
    tickets = [(srv.submit(sc), sc) for sc in [big[0], *small, big[1]]]
    srv.wait_idle(60000)
    for t, sc in tickets:
        assert srv.poll(t).state == _abi.REQ_DONE
        s = gpu_scene(sc)
        s.step(sc["frames"])
        s.sync()
        assert np.isfinite(srv.result(t)).all()
        assert_bit_equal(srv.result(t), s.download(_abi.DENSITY), f"N={sc['size'] - 2}")
        s.close()
    srv.close()
