"""A strip of the exact mode that gives up waiting for the one above it: no poll
allowed (eqf_ctx_set_wait_limit(0)) makes the second strip give up in its first
block, every kernel ends as always, and everything that hands the scene's fields
out says so until they are uploaded again."""
import time

import numpy as np
import pytest

from equilibrium_amd import _abi, scenes
from helpers import FIELD_NAMES, assert_bit_equal, download_all, gpu_scene

pytestmark = pytest.mark.gpu


def _scene(ctx, N=500, seed=1):  # nine strips
    p = _abi.default_params()
    p.size, p.delta_t, p.viscosity, p.diffusion, p.gs_iters, p.pressure_iters = N + 2, 0.1, 1e-5, 1e-5, 20, 20
    s = _abi.Scene(p, ctx)
    rng = np.random.default_rng(seed)
    fields = [(rng.standard_normal((N + 2) ** 2) * 0.05).astype(np.float32) for _ in FIELD_NAMES]
    for i, f in enumerate(fields):
        s.upload(i, f)
    return s, fields


def _fails(call):
    with pytest.raises(_abi.EqfError) as ei:
        call()
    assert ei.value.code == _abi.EQF_EDEVICE and "gave up" in str(ei.value)


def _stepped(fields, N=500):
    ctx = _abi.Context(0)
    s, _ = _scene(ctx, N)
    for i, f in enumerate(fields):
        s.upload(i, f)
    s.step(2)
    s.sync()
    d = download_all(s)
    s.close()
    ctx.close()
    return d


def _heals(ctx, s, fields):
    """Valid again field by field, and steps as a scene that never failed."""
    ctx.set_wait_limit(1 << 22)
    for i, f in enumerate(fields):
        _fails(s.sync)
        s.upload(i, f)
        assert_bit_equal(s.download(i), f, FIELD_NAMES[i])
    s.step(1)
    s.step(1)
    s.sync()
    want = _stepped(fields)
    for k, v in download_all(s).items():
        assert_bit_equal(v, want[k], k)


def test_scene_reports_until_its_fields_are_uploaded():
    print("[case] gave up: scene", flush=True)
    ctx = _abi.Context(0)
    s, fields = _scene(ctx)
    snap = _abi.Snapshot(s, depth=2, with_rgba=True)
    snap.capture(0)
    assert snap.acquire()[0] == 0  # before the failure
    snap.release()
    ctx.set_wait_limit(0)
    s.step(2)  # kernel by kernel, then the graph
    snap.capture(1)
    _fails(lambda: s.download(_abi.DENSITY))
    _fails(s.sync)
    _fails(s.render_rgba)
    _fails(s.render_rgba_noalloc)
    _fails(snap.acquire)
    snap.release()
    snap.capture(2)
    _fails(snap.acquire)
    snap.release()
    c = s.clone()
    _fails(lambda: c.download(_abi.VX))
    c.close()
    _heals(ctx, s, fields)
    snap.capture(3)
    assert snap.acquire()[0] == 3
    snap.capture(4)
    s.close()  # a ring keeps its captures
    snap.release()
    assert snap.acquire()[0] == 4
    snap.release()
    snap.close()
    ctx.close()


def test_a_step_makes_every_field_invalid_again():
    print("[case] gave up: partial upload", flush=True)
    ctx = _abi.Context(0)
    s, fields = _scene(ctx)
    ctx.set_wait_limit(0)
    s.step(1)
    ctx.set_wait_limit(1 << 22)
    s.upload(_abi.DENSITY, fields[0])
    assert_bit_equal(s.download(_abi.DENSITY), fields[0], "density")
    s.step(1)
    _fails(lambda: s.download(_abi.DENSITY))
    _heals(ctx, s, fields)
    s.close()
    ctx.close()


def test_batch_leaves_the_failure_to_its_scenes():
    print("[case] gave up: batch", flush=True)
    ctx = _abi.Context(0)
    pairs = [_scene(ctx, 500, k) for k in (2, 3)]
    b = _abi.Batch([s for s, _ in pairs], ctx)
    ctx.set_wait_limit(0)
    b.step(2)
    _fails(b.sync)
    _fails(lambda: pairs[0][0].download(_abi.VX))
    b.step(1)
    b.close()
    for s, fields in pairs:
        _fails(lambda: s.download(_abi.VX))
        _heals(ctx, s, fields)
        ctx.set_wait_limit(0)
    for s, _ in pairs:
        s.close()
    ctx.close()


def _until(srv, t, states):
    for _ in range(20000):
        st = srv.poll(t)
        if st.state in states:
            return st
        time.sleep(0.001)
    raise AssertionError(f"ticket {t} still in state {st.state}")


def test_served_request_fails_in_the_frame_that_gave_up():
    """The failure in a request's only (so last) frame is its own; the lane goes on
    with the next requests, and a cancelled one beside it is not held up."""
    print("[case] gave up: server", flush=True)
    ctx = _abi.Context(0)
    srv = _abi.Server(4 << 30, ctx=ctx)
    sc = [scenes.stam_scene(500, scenes.derive_seed(60, i), iters=20, frames=1 + i, n_rects=2) for i in range(3)]
    small = scenes.stam_scene(60, scenes.derive_seed(61), iters=20, frames=3)  # one lane further
    ended = (_abi.REQ_DONE, _abi.REQ_FAILED, _abi.REQ_CANCELLED)
    ctx.set_wait_limit(0)
    ts = [srv.submit(s, keep_velocity=True) for s in sc]
    for t in ts:
        st = _until(srv, t, ended)
        assert st.state == _abi.REQ_FAILED and st.frames_done == 0
        with pytest.raises(_abi.EqfError):
            srv.result(t)
        srv.release(t)
    ctx.set_wait_limit(1 << 22)
    ts = [srv.submit(s, keep_velocity=True) for s in sc + [small]]
    for t, s in zip(ts, sc + [small]):
        assert _until(srv, t, ended).state == _abi.REQ_DONE
        g = gpu_scene(s)
        g.step(s["frames"])
        g.sync()
        for f in (_abi.DENSITY, _abi.VX, _abi.VY):
            assert_bit_equal(srv.result(t, f), g.download(f), f"N={s['size'] - 2} field {f}")
        g.close()
    srv.close()
    ctx.close()
