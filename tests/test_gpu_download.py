"""Downloads through the context's pinned chunks: every remainder of a chunk,
several chunks, and several threads at once (more than buffers are kept)."""
import threading

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
