"""Steps between changes of parameters, sources, iteration counts and obstacles:
against the oracle bit for bit, and without a wait where only values change."""
import time

import numpy as np
import pytest

import oracle
from equilibrium_amd import _abi, scenes
from helpers import FIELD_NAMES, assert_state_equal, download_all, oracle_state

pytestmark = pytest.mark.gpu


def _params(S, mode, iters=6, press=9):
    p = _abi.default_params()
    p.size, p.gs_mode, p.gs_iters, p.pressure_iters = S, mode, iters, press
    p.delta_t, p.viscosity, p.diffusion = 0.1, 2.0 / S ** 2, 1.0 / S ** 2
    return p


@pytest.mark.parametrize("S", [30, 140])
@pytest.mark.parametrize("mode", [_abi.GS_WAVEFRONT, _abi.GS_REDBLACK])
def test_changes_between_steps_equal_oracle(S, mode):
    print(f"[case] changes S={S} mode={mode}", flush=True)
    rng = np.random.default_rng(S)
    p = _params(S, mode)
    s, st, src = _abi.Scene(p), oracle.State(S), {}
    m = (rng.random((S, S)) >= 0.05).astype(np.uint8)
    m[0] = m[-1] = 0
    m[:, 0] = m[:, -1] = 0
    s.set_mask(m.ravel())
    st.mask = m.ravel().copy()
    for i, k in enumerate(FIELD_NAMES):
        f = (rng.standard_normal(S * S) * (0.05 if k.startswith("v") else 1.0)).astype(np.float32)
        s.upload(i, f)
        st.f[k] = f.copy()
    order = oracle.RB if mode == _abi.GS_REDBLACK else oracle.LEX

    def go(n, label, **kw):
        for k, v in kw.items():
            setattr(p, k, v)
        if kw:
            s.set_params(p)
        for _ in range(n):
            s.step(1)
        st.run(p.delta_t, p.diffusion, p.viscosity, p.gs_iters, n, press_iters=p.pressure_iters, order=order,
               src_d=src.get(0), src_u=src.get(2), src_v=src.get(3))
        s.sync()
        assert_state_equal(download_all(s), st, label)

    def source(field, on):
        a = (rng.standard_normal(S * S) * 0.01).astype(np.float32) if on else None
        s.set_frame_source(field, a)
        src[field] = a

    go(3, "start")
    go(2, "dt", delta_t=0.07)  # the graph's frames
    go(1, "viscosity", viscosity=0.0)
    go(2, "diffusion", diffusion=0.0, viscosity=0.0)
    go(2, "dt alone", delta_t=0.03)
    source(_abi.DENSITY, True)
    go(3, "a source")
    source(_abi.DENSITY, True)
    go(1, "its amounts")
    source(_abi.VX, True)
    go(2, "two sources", delta_t=0.05)
    source(_abi.DENSITY, False)
    go(2, "one source")
    source(_abi.VX, False)
    go(2, "no source")
    go(2, "sweeps", gs_iters=25, pressure_iters=4)
    m[5:9, 6:11] = 0
    s.set_mask(m.ravel())
    st.mask = m.ravel().copy()
    go(2, "mask")
    m[:, 3] = 0  # a column without fluid
    s.set_mask(m.ravel())
    st.mask = m.ravel().copy()
    go(2, "walled column", delta_t=0.1)
    s.close()


@pytest.mark.parametrize("mode", [_abi.GS_WAVEFRONT, _abi.GS_REDBLACK])
def test_parameter_changes_do_not_wait_for_queued_frames(mode):
    print(f"[case] changes without a wait mode={mode}", flush=True)
    p = _params(1026, mode, 40, 40)
    s = _abi.Scene(p)
    s.step(3)
    s.sync()
    t0 = time.perf_counter()
    s.step(120)  # 0.1 to 0.3 s of frames
    t1 = time.perf_counter()
    for k in range(3):
        p.delta_t, p.viscosity = 0.09 + 0.01 * k, 1e-6 * k
        s.set_params(p)
        s.step(1)
    t2 = time.perf_counter()
    s.sync()
    t3 = time.perf_counter()
    print(f"[changes] queued in {1e3 * (t1 - t0):.1f} ms, changed in {1e3 * (t2 - t1):.1f}, done after {1e3 * (t3 - t0):.1f}",
          flush=True)
    assert t2 - t1 < 0.2 * (t3 - t0)
    s.close()


@pytest.mark.parametrize("mode,iters", [(_abi.GS_WAVEFRONT, 30000), (_abi.GS_REDBLACK, 9000)])
def test_more_launches_than_a_graph_holds_equal_oracle(mode, iters):
    """Frames of more than 4096 launches run kernel by kernel."""
    print(f"[case] long solves mode={mode} {iters}", flush=True)
    S = 6
    p = _params(S, mode, iters, iters)
    s, st = _abi.Scene(p), oracle.State(S)
    rng = np.random.default_rng(9)
    st.mask = s.get_mask()
    for i, k in enumerate(FIELD_NAMES):
        f = rng.standard_normal(S * S).astype(np.float32)
        s.upload(i, f)
        st.f[k] = f.copy()
    s.step(3)
    s.sync()
    st.run(p.delta_t, p.diffusion, p.viscosity, iters, 3, press_iters=iters,
           order=oracle.RB if mode == _abi.GS_REDBLACK else oracle.LEX)
    assert_state_equal(download_all(s), st, "long solves")
    s.close()


def test_a_batch_steps_scenes_whose_context_is_gone():
    """A batch belongs to its own context; what its scenes need of theirs they hold."""
    print("[case] scenes of a context that is destroyed", flush=True)
    sc = scenes.stam_scene(70, scenes.derive_seed(65), iters=5, frames=2, n_rects=1)
    a, b = _abi.Context(0), _abi.Context(0)
    s = _abi.Scene(scenes.scene_params(sc), a)
    scenes.apply_to_scene(s, sc)
    batch = _abi.Batch([s], b)
    a.close()
    batch.step(1)
    batch.step(1)
    batch.sync()
    st = oracle_state(sc)
    st.run(sc["dt"], sc["diffusion"], sc["viscosity"], sc["iters"], 2, src_d=sc["src_d"], src_u=sc["src_u"],
           src_v=sc["src_v"])
    assert_state_equal(download_all(s), st, "context gone")
    batch.close()
    s.close()
    b.close()
