"""The GPU BVH build where its schedule changes, against the host build: sets
around the size that one wave finishes alone (option bvh_small: 128 by default,
256 at most; a lane of that wave holds up to four items) and around a chunk of
the levels above (1024 items), alone and several in one scene."""
import numpy as np
import pytest

from barnacle_amd import configs, native, scene
from test_gpu_bvh import boxes, scene_blas

pytestmark = pytest.mark.gpu
KINDS = ["uniform", "clustered", "signed_zeros", "flat", "one_point", "skewed"]


@pytest.mark.parametrize("small", [128, 200, 256, 512])
@pytest.mark.parametrize("kind", KINDS)
def test_borders(ctx, kind, small):
    ctx.set_option("bvh_small", small)
    try:
        for n in (4, 5, 64, 65, 127, 128, 129, 192, 193, 200, 201, 255, 256, 257, 1023, 1024, 1025, 2047, 2048, 2049):
            print(f"{kind} {n}, bvh_small {small}", flush=True)
            b = boxes(kind, n, seed=small + n)
            hn, hp = native.bvh_build(b)
            gn, gp = ctx.bvh_build(b)
            assert gn.tobytes() == hn.tobytes() and np.array_equal(gp, hp), n
    finally:
        ctx.set_option("bvh_small", 128)


@pytest.mark.parametrize("small", [128, 256])
def test_sets_of_both_sizes_in_one_build(ctx, small):
    info = configs.cornell_box(16, 16, 1, 2)
    rng = np.random.default_rng(small)
    for n in (1, 127, 2000, 128, 129, 3, 255, 257, 1025, 256):
        v = (rng.uniform(100, 400, (n, 1, 3)) * [1, 1, -1] + rng.uniform(-9, 9, (n, 3, 3))).astype(np.float32)
        info["primitives"].append({"type": "mesh", "vertices": v.reshape(-1),
                                   "indices": np.arange(3 * n, dtype=np.int32)})
        info["instances"].append({"primitive": len(info["primitives"]) - 1, "material": 0})
        info["nodes"][0]["instances"].append(len(info["instances"]) - 1)
    sc = scene.load_scene(info)
    ctx.set_option("bvh_small", small)
    try:
        dg, bg = scene_blas(ctx, sc, 1)
        dh, bh = scene_blas(ctx, sc, 0)
    finally:
        ctx.set_option("bvh_small", 128)
    assert len(bg) == len(bh) and all(x == y for x, y in zip(bg, bh))
    p = sc.pt_params()
    assert np.array_equal(dg.render_pt(p).view(np.int32), dh.render_pt(p).view(np.int32))
    dg.release()
    dh.release()
