"""Small exact scenes in batches of many: whole solves in registers, a wave for up to
four of them.  Random fields and walls at the edges of the size classes (16, 32, 48, 64
and 66 rows), all sweep counts side by side, against the oracle bit for bit."""
import numpy as np
import pytest

import oracle
from equilibrium_amd import _abi
from helpers import FIELD_NAMES, assert_state_equal, download_all

pytestmark = pytest.mark.gpu

SIZES = [3, 4, 5, 15, 16, 17, 18, 31, 32, 33, 34, 47, 48, 49, 50, 63, 64, 65, 66, 67, 90]


def _scene(S, iters, press, walls, rng, full=()):
    m = (rng.random((S, S)) >= walls).astype(np.uint8)
    for v in full:
        if 0 < abs(v) < S - 1:
            if v > 0:
                m[:, v] = 0
            else:
                m[-v, :] = 0
    m[0] = m[-1] = 0
    m[:, 0] = m[:, -1] = 0
    p = _abi.default_params()
    p.size, p.delta_t, p.viscosity, p.diffusion = S, 0.1, 3.0 / (S - 2) ** 2, 1.0 / (S - 2) ** 2
    p.gs_iters, p.pressure_iters = iters, press
    s = _abi.Scene(p)
    s.set_mask(m.ravel())
    st = oracle.State(S)
    st.mask = m.ravel().copy()
    for i, k in enumerate(FIELD_NAMES):
        f = (rng.standard_normal(S * S) * (0.05 if k.startswith("v") else 1.0)).astype(np.float32)
        s.upload(i, f)
        st.f[k] = f.copy()
    return s, st, lambda n: st.run(p.delta_t, p.diffusion, p.viscosity, iters, n, press_iters=press)


def _check(specs, seed, walls=0.1, full=()):
    rng = np.random.default_rng(seed)
    trio = [_scene(*sp, walls, rng, full) for sp in specs]
    b = _abi.Batch([s for s, _, _ in trio])
    b.step(1)  # kernel by kernel, then the graph
    b.step(1)
    b.sync()
    for (s, st, run), sp in zip(trio, specs):
        run(2)
        assert_state_equal(download_all(s), st, f"{sp}")
    b.close()
    for s, _, _ in trio:
        s.close()


@pytest.mark.parametrize("walls,full", [(0.0, ()), (0.15, ()), (0.5, ()), (0.05, (1, -1)), (0.05, (2, 9, -30, 46, -64)), (0.1, (64, -63))])
def test_many_small_scenes_equal_oracle(walls, full):
    """280 scenes of every size beside each other: the groups of a wave differ in size
    and sweep counts (0 too), and larger scenes take the strips."""
    print(f"[case] small scenes walls={walls} full={full}", flush=True)
    specs = [(SIZES[(i * 5) % len(SIZES)], (i * 7) % 23, (3 + i * 11) % 22) for i in range(310)]
    _check(specs, 5, walls, full)


@pytest.mark.parametrize("S", [3, 16, 17, 32, 33, 48, 49, 64, 65, 66])
def test_one_size_equals_oracle(S):
    print(f"[case] small scenes S={S}", flush=True)
    _check([(S, 20, 20 + i % 3) for i in range(257)], S)


@pytest.mark.parametrize("n", [255, 256])  # either side of the rule
def test_either_side_of_the_rule_equals_oracle(n):
    print(f"[case] {n} small scenes", flush=True)
    _check([(30 + i % 37, 1 + i % 5, 2) for i in range(n)] + [(100, 4, 4)], 77)


def test_more_than_a_round_of_sweeps_equals_oracle():
    print("[case] small scenes, many sweeps", flush=True)
    _check([(10 + i % 57, 61, 45) for i in range(260)], 78)
