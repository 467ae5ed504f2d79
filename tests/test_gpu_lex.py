"""The lexicographic lin_solve on the GPU at the edges of its split: strips of
63 rows that move up a row per sweep, four waves of up to five sweeps, rounds of
20 sweeps, blocks of 8 steps.  Random fields and walls, frames of the whole step
against the oracle, bit for bit."""
import numpy as np
import pytest

import oracle
from equilibrium_amd import _abi
from helpers import FIELD_NAMES, assert_state_equal, download_all

pytestmark = pytest.mark.gpu


def _pair(S, iters, press, walls, seed, full=()):
    """A scene with random fields and walls on the GPU and in the oracle;
    `full`: rows / columns (>= 0: column, < 0: row -v) walled from side to side."""
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
    p.size, p.delta_t, p.viscosity, p.diffusion = S, 0.1, 3.0 / (S - 2 or 1) ** 2, 1.0 / (S - 2 or 1) ** 2
    p.gs_iters, p.pressure_iters = iters, press
    s = _abi.Scene(p)
    s.set_mask(m.ravel())
    st = oracle.State(S)
    st.mask = m.ravel().copy()
    for i, k in enumerate(FIELD_NAMES):
        f = (rng.standard_normal(S * S) * (0.05 if k.startswith("v") else 1.0)).astype(np.float32)
        s.upload(i, f)
        st.f[k] = f.copy()
    run = lambda n: st.run(p.delta_t, p.diffusion, p.viscosity, iters, n, press_iters=press)
    return s, st, run


@pytest.mark.parametrize("S,iters,press", [
    (3, 20, 20), (4, 1, 2), (22, 3, 4),      # one cell; fewer sweeps than waves
    (44, 20, 20), (45, 20, 20),              # K + S - 1 = 63 / 64 rows: one strip, two
    (46, 20, 20), (107, 20, 20), (108, 20, 20),
    (64, 5, 7), (65, 13, 16), (66, 19, 6),   # uneven sweeps per wave
    (109, 20, 20), (110, 20, 21),            # two strips, three; a second round of one sweep more
    (131, 41, 25), (258, 20, 40),            # three rounds, two
    (515, 20, 5), (1026, 4, 1),              # many strips, the largest size
])
@pytest.mark.parametrize("walls", [0.0, 0.1])
def test_split_edges_equal_oracle(S, iters, press, walls):
    print(f"[case] lex S={S} iters={iters} press={press} walls={walls}", flush=True)
    s, st, run = _pair(S, iters, press, walls, S * 1000 + iters)
    n = 2 if S < 500 else 1
    s.step(n)
    s.sync()
    run(n)
    assert_state_equal(download_all(s), st, f"S={S}")
    s.close()


@pytest.mark.parametrize("full", [(1,), (-1,), (30, -40), (68, -68)])
def test_ring_cells_without_fluid_neighbours_equal_oracle(full):
    """Rows / columns without a NoWall cell: their ring cells keep their values
    (no Passive copy), by the general selectors instead of the masks."""
    print(f"[case] lex walled rows / columns {full}", flush=True)
    s, st, run = _pair(70, 6, 9, 0.05, 5, full)
    s.step(2)
    s.sync()
    run(2)
    assert_state_equal(download_all(s), st, f"walled {full}")
    s.close()


def test_batch_of_different_iteration_counts_equals_oracle():
    """One launch covers scenes whose solves have 0, 1 and several rounds."""
    print("[case] lex batch of iteration counts", flush=True)
    specs = [(40, 0, 3), (90, 25, 0), (70, 1, 20), (130, 20, 45), (33, 60, 2), (200, 7, 7)]
    trio = [_pair(S, it, pr, 0.05, 70 + i) for i, (S, it, pr) in enumerate(specs)]
    b = _abi.Batch([s for s, _, _ in trio])
    for n in (1, 2):  # kernel by kernel, then the replayed graph too
        b.step(n)
    b.sync()
    for (s, st, run), spec in zip(trio, specs):
        run(3)
        assert_state_equal(download_all(s), st, f"{spec}")
    b.close()
    for s, _, _ in trio:
        s.close()


# fewer strips than CUs (eight waves of sweeps each); more (four); more, long ones (eight); many (four)
@pytest.mark.parametrize("n,step", [(20, 13), (90, 13), (40, 40), (90, 40)])
def test_batches_either_side_of_the_wave_count_equal_oracle(n, step):
    print(f"[case] lex batch of {n}, {step}", flush=True)
    specs = [(20 + step * (i % 9), 1 + i % 23, 1 + (7 * i) % 22) for i in range(n)]
    trio = [_pair(S, it, pr, 0.05, 900 + i) for i, (S, it, pr) in enumerate(specs)]
    b = _abi.Batch([s for s, _, _ in trio])
    b.step(2)
    b.sync()
    for (s, st, run), spec in zip(trio, specs):
        run(2)
        assert_state_equal(download_all(s), st, f"{spec}")
    b.close()
    for s, _, _ in trio:
        s.close()
