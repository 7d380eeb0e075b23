"""A round whose paths all fit the slots starts them in its first iteration and
runs exactly its depth of iterations, eagerly or as one captured graph (up to
64 iterations); a round of more paths than slots refills them and is watched
by the host.  Films are the same, bit for bit, and a second use of the same
buffers starts from black again."""
import numpy as np
import pytest

from barnacle_amd import configs, scene

pytestmark = pytest.mark.gpu


@pytest.mark.parametrize("depth", [0, 1, 2, 3, 64, 65])
@pytest.mark.parametrize("spp", [0, 1, 3])
def test_rounds_at_once_equal_streamed_rounds(ctx, depth, spp):
    sc = scene.load_scene(configs.config1(width=61, height=43, spp=spp, max_depth=depth, freq=6))
    ds = ctx.scene(sc)
    p = sc.pt_params()
    print(f"depth {depth}, {spp} samples", flush=True)
    try:
        ctx.set_option("window_paths", 1 << 20)
        ctx.set_option("chunk_slots", 1024)                 # fewer slots than a sample's paths
        ref = ds.render_pt(p)
        ctx.set_option("window_paths", 0)
        ctx.set_option("chunk_slots", 64 << 20)
        at_once = [ds.render_pt(p), ds.render_pt(p)]
        batched = [f for _ in range(3) for f in ctx.render_batch([(ds, p), (ds, p)])[0]]
    finally:
        ctx.set_option("window_paths", 0)
        ctx.set_option("chunk_slots", 64 << 20)
        ds.release()
    assert (ref != 0).any() == (depth > 0 and spp > 0)
    for film in at_once + batched:
        assert np.array_equal(film.view(np.int32), ref.view(np.int32))
