"""Steps one workload, for a profiler: python3 profiles/frames.py WORKLOAD FRAMES

mix       512 scenes, N in {64, 128, 256, 512}, 20 sweeps, exact, one batch
rbmix     the same in red-black order
n1024     one exact scene, N=1024, 20 sweeps
n30       one exact scene, N=30, 16 sweeps
n4096     one red-black scene, N=4096, 40 sweeps, 16 rectangles
small     2048 exact scenes of N=62, 20 sweeps, one batch
"""
import os
import sys

sys.path.insert(0, os.path.join(os.path.dirname(os.path.abspath(__file__)), ".."))
from equilibrium_amd import _abi, scenes  # noqa: E402


def main(what, frames):
    mode = _abi.GS_REDBLACK if what in ("rbmix", "n4096") else _abi.GS_WAVEFRONT
    if what in ("mix", "rbmix"):
        scs = scenes.batched_mix(frames=frames)
    elif what == "small":
        scs = [scenes.stam_scene(62, scenes.derive_seed(i)) for i in range(2048)]
    else:
        scs = [{"n1024": scenes.single_1024, "n4096": scenes.redblack_scene,
                "n30": lambda: scenes.stam_scene(30, scenes.derive_seed(1), iters=16)}[what]()]
    hs = []
    for sc in scs:
        h = _abi.Scene(scenes.scene_params(sc, mode))
        scenes.apply_to_scene(h, sc)
        hs.append(h)
    run = _abi.Batch(hs) if len(hs) > 1 else hs[0]
    run.step(frames)
    run.sync()
    print(what, len(hs), "scenes", frames, "frames", flush=True)


if __name__ == "__main__":
    main(sys.argv[1], int(sys.argv[2]))
