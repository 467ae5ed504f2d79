"""A strip of the exact mode that gives up waiting for the one above it: no poll
allowed (eqf_ctx_set_wait_limit(0)) makes the second strip give up in its first
block, every kernel ends as always, and everything that hands the scene's fields
out says so until they are uploaded again."""
import numpy as np
import pytest

from equilibrium_amd import _abi
from helpers import FIELD_NAMES, assert_bit_equal, download_all

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
