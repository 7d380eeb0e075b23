"""The GPU BVH build at the edges of what it takes: trees as deep as the depth
limit, whose last leaf holds what a node's int8 count can hold and no more."""
import numpy as np
import pytest

from barnacle_amd import configs, native, scene

pytestmark = pytest.mark.gpu
BN_E_CAPACITY = -5


def point_boxes(x):
    p = np.zeros((len(x), 3), np.float32)
    p[:, 0] = x
    return np.concatenate([p, p], 1)


def peeled(kind, n):
    """n points that stay together in the leaf at depth 64, behind 64 that leave one a level."""
    if kind == "powers_of_13":                  # the 67 points 13^-33 .. 13^33: the last three stay too
        return point_boxes(np.concatenate([13.0 ** np.arange(-33, 34), np.zeros(n - 3)]))
    return point_boxes(np.concatenate([np.zeros(n), 2.0 ** (-120 + 3.75 * np.arange(64))]))


@pytest.mark.parametrize("small", [128, 512])
@pytest.mark.parametrize("kind", ["powers_of_13", "powers_of_2"])
@pytest.mark.parametrize("n", [100, 127, 128, 256, 257, 300, 3003, 5000])
def test_leaf_at_the_depth_limit(ctx, kind, n, small):
    b = peeled(kind, n)
    print(f"{kind} {n}, bvh_small {small}", flush=True)
    ctx.set_option("bvh_small", small)
    try:
        if n <= 127:
            hn, hp = native.bvh_build(b)
            gn, gp = ctx.bvh_build(b)
            assert gn.tobytes() == hn.tobytes() and np.array_equal(gp, hp)
            assert gn["count"][gn["is_leaf"] != 0].max() == n
        else:
            for build in (native.bvh_build, ctx.bvh_build):
                with pytest.raises(native.BarnacleError, match="int8 count") as e:
                    build(b)
                assert e.value.code == BN_E_CAPACITY
        after = point_boxes(np.arange(1000.0))
        assert ctx.bvh_build(after)[0].tobytes() == native.bvh_build(after)[0].tobytes()
    finally:
        ctx.set_option("bvh_small", 128)


def test_scene_with_such_a_mesh_is_refused(ctx):
    x = peeled("powers_of_13", 3003)[:, :3]
    info = configs.cornell_box(16, 16, 1, 2)
    info["primitives"][0] = {"type": "mesh", "vertices": x.reshape(-1),
                             "indices": np.repeat(np.arange(len(x), dtype=np.int32), 3)}
    with pytest.raises(native.BarnacleError, match="int8 count") as e:
        ctx.scene(scene.load_scene(info))
    assert e.value.code == BN_E_CAPACITY


def one_far_away(n):
    """Finite boxes, of which one has a centroid that overflows: the extent of
    the centroids is infinite, all items of a node fall in its first bin, and
    every node down to the depth limit has a right child without items."""
    rng = np.random.default_rng(n)
    lo = rng.uniform(-9, 9, (n, 3))
    b = np.concatenate([lo, lo + 1], 1).astype(np.float32)
    b[n // 2, [0, 3]] = 3e38
    return b


@pytest.mark.parametrize("n", [4, 65, 100, 127])
def test_nodes_without_items(ctx, n):
    b = one_far_away(n)
    print(f"{n} boxes", flush=True)
    hn, hp = native.bvh_build(b)
    gn, gp = ctx.bvh_build(b)
    assert gn.tobytes() == hn.tobytes() and np.array_equal(gp, hp)
    assert len(gn) == (1 if n == 4 else 2 * 64 + 1)


@pytest.mark.parametrize("n", [128, 129, 3000])
def test_more_such_boxes_than_a_leaf_holds(ctx, n):
    for build in (native.bvh_build, ctx.bvh_build):
        with pytest.raises(native.BarnacleError, match="int8 count") as e:
            build(one_far_away(n))
        assert e.value.code == BN_E_CAPACITY


@pytest.mark.parametrize("n", [5, 20, 63, 64])
def test_trees_of_more_nodes_than_two_an_item(ctx, n):
    """129 nodes for at most 64 items: the GPU build has room for two nodes an
    item, refuses, and is as good as new."""
    with pytest.raises(native.BarnacleError, match="node count"):
        ctx.bvh_build(one_far_away(n))
    after = np.concatenate([one_far_away(4), point_boxes(np.arange(300.0))])
    with pytest.raises(native.BarnacleError, match="int8 count"):
        ctx.bvh_build(after)
    assert ctx.bvh_build(after[4:])[0].tobytes() == native.bvh_build(after[4:])[0].tobytes()
