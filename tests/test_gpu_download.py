"""Downloads through the context's pinned chunks: every remainder of a chunk,
several chunks, and several threads at once (more than buffers are kept)."""
import ctypes
import threading
import time

import numpy as np
import pytest

from equilibrium_amd import _abi

pytestmark = pytest.mark.gpu


def _scene(S, seed):
    p = _abi.default_params()
    p.size, p.gs_mode = S, _abi.GS_REDBLACK
    s = _abi.Scene(p)
    a = np.random.default_rng(seed).standard_normal(S * S).astype(np.float32)
    s.upload(_abi.VX, a)
    return s, a


# chunks of at most 2 MB: 724 * 724 * 4 is just below, 725 * 725 * 4 just above
@pytest.mark.parametrize("S", [3, 66, 724, 725, 1025, 1449, 2051])
def test_download_returns_what_was_uploaded(S):
    s, a = _scene(S, S)
    for _ in range(3):
        assert np.array_equal(s.download(_abi.VX), a)
    s.close()


def test_downloads_from_several_threads():
    pairs = [_scene(S, S) for S in (66, 130, 725, 1100, 300, 1449, 900, 64)]
    bad = []

    def work(s, a):
        for _ in range(10):
            if not np.array_equal(s.download(_abi.VX), a):
                bad.append(len(a))

    ts = [threading.Thread(target=work, args=p) for p in pairs]
    for t in ts:
        t.start()
    for t in ts:
        t.join()
    assert not bad
    for s, _ in pairs:
        s.close()


class _Mem:
    """Memory of the HIP runtime: pinned, or the device's."""

    def __init__(self, nbytes, pinned):
        self.hip = ctypes.CDLL("libamdhip64.so")
        self.pinned, p = pinned, ctypes.c_void_p()
        n = ctypes.c_size_t(nbytes)
        assert (self.hip.hipHostMalloc(ctypes.byref(p), n, 0) if pinned else self.hip.hipMalloc(ctypes.byref(p), n)) == 0
        self.p, self.nbytes = p, nbytes

    def read(self):
        a = np.empty(self.nbytes // 4, np.float32)
        assert self.hip.hipMemcpy(a.ctypes.data_as(ctypes.c_void_p), self.p, ctypes.c_size_t(self.nbytes), 4) == 0
        return a

    def close(self):
        assert (self.hip.hipHostFree(self.p) if self.pinned else self.hip.hipFree(self.p)) == 0


@pytest.mark.parametrize("pinned", [True, False])
@pytest.mark.parametrize("S", [3, 725, 2051])
def test_download_into_memory_of_the_runtime(S, pinned):
    s, a = _scene(S, S)
    m = _Mem(4 * S * S, pinned)
    for _ in range(2):
        _abi.check(_abi.lib().eqf_download(s.h, _abi.VX, m.p))
        assert np.array_equal(m.read(), a)
    m.close()
    s.close()


def test_pinned_memory_takes_no_copy_by_the_host():
    """67 MB: 1.2 ms straight, 2.5 ms through the chunks."""
    S = 4098
    s, a = _scene(S, S)
    m, page = _Mem(4 * S * S, True), np.zeros(S * S, np.float32)

    def us(p):
        t = []
        for _ in range(9):
            t0 = time.perf_counter()
            _abi.check(_abi.lib().eqf_download(s.h, _abi.VX, p))
            t.append(time.perf_counter() - t0)
        return sorted(t)[4] * 1e6

    pinned, pageable = us(m.p), us(_abi.ptr(page))
    print(f"[download] pinned {pinned:.0f} us, pageable {pageable:.0f} us", flush=True)
    assert np.array_equal(m.read(), a) and np.array_equal(page, a)
    assert pinned < 0.75 * pageable
    m.close()
    s.close()
