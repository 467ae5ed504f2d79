"""Divergence, gradient and advection with their set_boundaries inside, at the
edges of their split (segments of 256 cells of a row, 64 to a lane group; rows
of 4, 8 and 16 waves and longer ones), with walls that cells take values from,
rows and columns without fluid (ring cells that keep theirs), and velocities
that reach the far edge (rows that stop).  Whole frames against the oracle, bit
for bit."""
import numpy as np
import pytest

import oracle
from equilibrium_amd import _abi
from helpers import FIELD_NAMES, assert_state_equal, download_all

pytestmark = pytest.mark.gpu


def _pair(N, mode, seed, walls=0.1, full=(), speed=1.0, iters=2, press=3):
    S = N + 2
    rng = np.random.default_rng(seed)
    m = (rng.random((S, S)) >= walls).astype(np.uint8)
    for v in full:
        if v >= 0:
            m[:, v] = 0
        else:
            m[-v, :] = 0
    m[0] = m[-1] = 0
    m[:, 0] = m[:, -1] = 0
    p = _abi.default_params()
    p.size, p.delta_t, p.viscosity, p.diffusion = S, 0.1, 1.0 / N ** 2, 0.5 / N ** 2
    p.gs_iters, p.pressure_iters, p.gs_mode = iters, press, mode
    s = _abi.Scene(p)
    s.set_mask(m.ravel())
    st = oracle.State(S)
    st.mask = m.ravel().copy()
    for i, k in enumerate(FIELD_NAMES):
        f = (rng.standard_normal(S * S) * (speed if k.startswith("v") else 1.0)).astype(np.float32)
        s.upload(i, f)
        st.f[k] = f.copy()
    order = oracle.RB if mode == _abi.GS_REDBLACK else oracle.LEX
    return s, st, lambda n: st.run(p.delta_t, p.diffusion, p.viscosity, iters, n, press_iters=press, order=order)


@pytest.mark.parametrize("N", [1, 2, 63, 64, 65, 128, 129, 192, 193, 255, 256, 257, 320, 449, 512, 513, 1024])
@pytest.mark.parametrize("mode", [_abi.GS_WAVEFRONT, _abi.GS_REDBLACK])
def test_segment_edges_equal_oracle(N, mode):
    print(f"[case] phases N={N} mode={mode}", flush=True)
    s, st, run = _pair(N, mode, N)
    s.step(2)
    s.sync()
    run(2)
    assert_state_equal(download_all(s), st, f"N={N}")
    s.close()


@pytest.mark.parametrize("N", [1025, 2048, 2049, 4097])  # 8 waves to a row, 16, rows in two passes
def test_long_rows_equal_oracle(N):
    print(f"[case] phases long rows N={N}", flush=True)
    s, st, run = _pair(N, _abi.GS_REDBLACK, N)
    s.step(1)
    s.sync()
    run(1)
    assert_state_equal(download_all(s), st, f"N={N}")
    s.close()


@pytest.mark.parametrize("full", [(1,), (70,), (-1,), (-70,), (1, 70, -1, -70), (35, -36)])
@pytest.mark.parametrize("mode", [_abi.GS_WAVEFRONT, _abi.GS_REDBLACK])
@pytest.mark.parametrize("speed", [0.0, 30.0])
def test_walled_rows_and_breaks_equal_oracle(full, mode, speed):
    print(f"[case] phases walled {full} mode={mode} speed={speed}", flush=True)
    s, st, run = _pair(70, mode, 7, 0.2, full, speed)
    s.step(2)
    s.sync()
    run(2)
    assert_state_equal(download_all(s), st, f"{full}")
    s.close()


@pytest.mark.parametrize("sizes", [(1100, 30, 256, 257, 700), (3071, 40)])
def test_batch_of_row_lengths_equals_oracle(sizes):
    """Short rows (a wave each) beside rows of several waves in one launch; with
    a scene of one ping-pong field in the batch the diffusions run apart."""
    print(f"[case] phases batch {sizes}", flush=True)
    trio = [_pair(N, _abi.GS_REDBLACK, N) for N in sizes]
    b = _abi.Batch([s for s, _, _ in trio])
    for n in (1, 1):
        b.step(n)
    b.sync()
    for (s, st, run), N in zip(trio, sizes):
        run(2)
        assert_state_equal(download_all(s), st, f"N={N}")
    b.close()
    for s, _, _ in trio:
        s.close()


@pytest.mark.parametrize("N", [128, 300])  # several tiles in both directions
@pytest.mark.parametrize("walls", [0.2, 0.5])
@pytest.mark.parametrize("tile,tsw", [(5, 5), (0, 8), (1, 6), (2, 4)])
def test_redblack_tile_halos_with_dense_walls(N, walls, tile, tsw):
    """Every sweep of a launch carries values across tiles through walls too."""
    print(f"[case] phases halo N={N} walls={walls} tile={tile} T={tsw}", flush=True)
    s, st, run = _pair(N, _abi.GS_REDBLACK, 11, walls, iters=20, press=17)
    s.set_tuning(tile, tsw)
    s.step(2)
    s.sync()
    run(2)
    assert_state_equal(download_all(s), st, f"N={N}")
    s.close()
