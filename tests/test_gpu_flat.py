"""Scenes are traversed by records of their nodes, those of at most 32 instances
through a list of their bounds in place of the TLAS: the same films and hits as the walk of the reference's
tree (the counting kernels), on both sides of the limit, for rays with zero
direction components (whose slab tests see NaNs: bounds in the plane of the
origin) and for a tree whose nodes do not contain their instances."""
import numpy as np
import pytest

from barnacle_amd import configs, scene
from test_gpu_upload import reupload

pytestmark = pytest.mark.gpu


def cubes(n, fov, integrator=None):
    info = configs.cornell_box(27, 21, 3, 5, boxes=False)
    info["integrator"] = integrator or info["integrator"]
    info["camera"]["fov"] = fov
    eye = info["transforms"][-1]["keyframes"][0]["translation"]
    info["primitives"].append({"type": "cube"})
    rng = np.random.default_rng(n)
    for k in range(n - len(info["instances"])):
        key = {"time": 0.0, "scale": [float(x) for x in rng.uniform(10, 60, 3)],
               "translation": [float(rng.uniform(50, 500)), float(rng.uniform(50, 500)), float(-rng.uniform(50, 500))]}
        if k % 3 == 0:                      # a face in the plane of the camera
            key["translation"][k % 2] = eye[k % 2] + key["scale"][k % 2]
        elif k % 3 == 1:
            key["rotation"] = [float(x) for x in rng.uniform(-1, 1, 3)]
        info["instances"].append({"primitive": len(info["primitives"]) - 1, "material": k % 3})
        info["transforms"].append({"keyframes": [key]})
        info["nodes"].append({"instances": [len(info["instances"]) - 1], "transform": len(info["transforms"]) - 1})
        info["nodes"][0]["children"].append(len(info["nodes"]) - 1)
    return scene.load_scene(info)


def same(a, b):
    return np.array_equal(np.asarray(a).view(np.int32), np.asarray(b).view(np.int32))


@pytest.mark.parametrize("fov", [39.3, 0.0])
@pytest.mark.parametrize("n", [6, 7, 20, 31, 32, 33, 40])
@pytest.mark.parametrize("records", [1, 0])
def test_few_instances_equal_the_tree_walk(ctx, orc, n, fov, records):
    print(f"{n} instances, fov {fov}, records {records}", flush=True)
    sc = cubes(n, fov)
    ctx.set_option("records", records)
    try:
        ds = ctx.scene(sc)
    finally:
        ctx.set_option("records", 1)
    p = sc.pt_params()
    walked, _ = ds.render_pt(p, stats=True)
    assert same(ds.render_pt(p), walked)
    for film in ctx.render_batch([(ds, p), (ds, p)])[0]:
        assert same(film, walked)
    for got, want in zip(ds.first_hit(p, 0), orc.scene(sc).first_hit(p, 0)):
        assert same(got, want)
    for got, want in zip(ds.first_hit_noalloc(p, 1), orc.scene(sc).first_hit(p, 1)):
        assert same(got, want)
    ds.release()


def test_nodes_that_no_other_leads_to(ctx):
    from barnacle_amd.bvh_util import NODE_DTYPE
    sc = cubes(9, 0.0)
    built = ctx.scene(sc)
    export, export_blas = built.export, built.export_blas
    stray = np.zeros(1, NODE_DTYPE)
    stray["split_axis"], stray["right_or_offset"] = 1, 1 << 28
    leaf = np.zeros(1, NODE_DTYPE)
    leaf["is_leaf"], leaf["count"], leaf["pmin"], leaf["pmax"] = 1, 9, -1e4, 1e4

    def more(ex, key, node):
        ex[key] = np.concatenate([ex[key], node])
        return ex

    built.export = lambda: more(export(), "tlas", leaf)
    built.export_blas = lambda prim: more(export_blas(prim), "nodes", stray)
    up, _ = reupload(ctx, sc, built)
    p = sc.pt_params()
    assert same(up.render_pt(p), built.render_pt(p))
    up.release()
    built.release()


@pytest.mark.parametrize("shrink", [0, 1, 2])
def test_tree_that_does_not_contain_its_instances(ctx, shrink):
    """An uploaded TLAS culls what its nodes leave out, whatever the bounds of
    the instances say."""
    sc = cubes(14, 39.3)
    built = ctx.scene(sc)
    export = built.export

    def cut():
        ex = export()
        node = ex["tlas"][min(shrink, len(ex["tlas"]) - 1)]
        node["pmin"][0] += np.float32(0.4) * (node["pmax"][0] - node["pmin"][0])
        return ex

    built.export = cut
    up, _ = reupload(ctx, sc, built)
    p = sc.pt_params()
    walked, _ = up.render_pt(p, stats=True)
    assert same(up.render_pt(p), walked)
    assert not same(walked, built.render_pt(p))
    up.release()
    built.release()


@pytest.mark.parametrize("change", ["instance", "root"])
def test_identity_instance_with_bounds_of_its_own(ctx, change):
    """An instance with an identity transform enters its BLAS without a test of
    the root only where the bounds of the two are the same."""
    sc = cubes(8, 39.3)
    built = ctx.scene(sc)
    if change == "instance":
        insts = built.export_instances()
        for rec in insts[:4]:
            rec.bounds[0] += np.float32(0.3) * np.float32(rec.bounds[3] - rec.bounds[0])
        built.export_instances = lambda: insts
    else:
        export_blas = built.export_blas

        def cut(prim):
            b = export_blas(prim)
            root = b["nodes"][0]
            root["pmin"][0] += np.float32(0.3) * (root["pmax"][0] - root["pmin"][0])
            return b

        built.export_blas = cut
    up, _ = reupload(ctx, sc, built)
    p = sc.pt_params()
    walked, _ = up.render_pt(p, stats=True)
    assert same(up.render_pt(p), walked)
    assert not same(walked, built.render_pt(p))
    up.release()
    built.release()


@pytest.mark.parametrize("sizes", [(7, 20, 32), (7, 40, 20)])
def test_mixed_batches_equal_plain_frames(ctx, sizes):
    """A batch round binds each ray's scene: lists where all its scenes have
    one, else trees; the same graph key must not stand for both."""
    ds = [ctx.scene(cubes(n, 39.3)) for n in sizes]
    ctx.set_option("records", 0)
    try:
        ds.append(ctx.scene(cubes(11, 39.3)))
    finally:
        ctx.set_option("records", 1)
    ps = [d.sc.pt_params() for d in ds]
    for pick in ((0, 1, 2), (0, 2), (1, 0), (0, 2), (0, 3), (0, 2)):
        for k, film in zip(pick, ctx.render_batch([(ds[k], ps[k]) for k in pick])[0]):
            assert same(film, ds[k].render_pt(ps[k], stats=True)[0])
    for d in ds:
        d.release()


@pytest.mark.parametrize("n", [20, 40])
def test_metropolis_waves_equal_the_wavefront(ctx, n):
    caustics = configs.caustic_scene(width=27, height=21, spp=2, max_depth=5, freq=4, n_bootstrap=512, n_chains=37)
    sc = cubes(n, 39.3, caustics["integrator"])
    ds = ctx.scene(sc)
    p = sc.mlt_params()
    out = []
    try:
        for waves in (0, 1 << 20):
            ctx.set_option("mlt_wave_chains", waves)
            film, st = ds.render_pssmlt(p)
            out.append((st["accepted"], ds.pssmlt_last(p)[1].copy(), film))
    finally:
        ctx.set_option("mlt_wave_chains", 20480)
    assert out[0][0] == out[1][0] and np.array_equal(out[0][1], out[1][1])
    assert np.allclose(out[0][2], out[1][2], rtol=1e-4, atol=1e-5, equal_nan=True)
    ds.release()


def test_leaves_of_many_triangles(ctx):
    """References of up to 127 triangles: an uploaded BLAS that is one leaf, and
    one whose leaves hold none."""
    from barnacle_amd.bvh_util import NODE_DTYPE
    sc = cubes(9, 39.3)
    built = ctx.scene(sc)
    export_blas = built.export_blas

    def one_leaf(prim):
        b = export_blas(prim)
        n = len(b["tri"].reshape(-1, 3))
        root = b["nodes"][0].copy()
        if n > 2:
            root["is_leaf"], root["right_or_offset"], root["count"] = 1, 0, n
            b["nodes"] = np.array([root], NODE_DTYPE)
        else:
            left = root.copy()
            left["is_leaf"], left["right_or_offset"], left["count"] = 1, 0, 0
            right = left.copy()
            right["count"] = n
            root["is_leaf"], root["right_or_offset"], root["split_axis"] = 0, 2, 1
            b["nodes"] = np.array([root, left, right], NODE_DTYPE)
        return b

    built.export_blas = one_leaf
    up, _ = reupload(ctx, sc, built)
    p = sc.pt_params()
    walked, _ = up.render_pt(p, stats=True)
    assert same(up.render_pt(p), walked)
    up.release()
    built.release()
