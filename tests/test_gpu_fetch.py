"""How rays reach the waves of a traversal: a queue that the grid's lanes hold
at once is dealt out (1 to 64 rays a wave), a longer one is fetched from
segments with a counter each.  Every ray is traced exactly once either way, so
the first hits equal the oracle's, bit for bit."""
import numpy as np
import pytest

from barnacle_amd import configs, scene

pytestmark = pytest.mark.gpu

# one wave and a ragged second; one ray a wave of 2048 and one more; 64 rays a
# wave of one block per CU (65536) and one more; the lanes of seven (458752) and
# one more
SIZES = [(1, 1), (65, 1), (2048, 1), (683, 3), (256, 256), (65537, 1), (1024, 448), (458753, 1)]


@pytest.mark.parametrize("blocks", [1, 7])
@pytest.mark.parametrize("size", SIZES)
def test_first_hits_of_every_queue_length(ctx, orc, size, blocks):
    w, h = size
    sc = scene.load_scene(configs.config1(width=w, height=h, spp=1, freq=8))
    p = sc.pt_params()
    print(f"first hits {w}x{h}, {blocks} blocks per CU", flush=True)
    ds = ctx.scene(sc)
    ctx.set_option("trace_blocks_per_cu", blocks)
    try:
        got = ds.first_hit(p)
    finally:
        ctx.set_option("trace_blocks_per_cu", 7)
        ds.release()
    ref = orc.scene(sc).first_hit(p)
    assert np.array_equal(got[0], ref[0]) and np.array_equal(got[1], ref[1])
    assert np.array_equal(got[2].view(np.int32), ref[2].view(np.int32))
